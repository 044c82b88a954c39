// FCHL19 representation, its VJP and its explicit Jacobian for gfx950.
// Replaces qml_lightning/cuda/fchl_cuda_kernel.cu:476-674 (forward), :1325-1714 (VJP),
// :676-1005 and :1007-1323 (Jacobian) of the reference.
//
// Layout: one wavefront (64 lanes, one workgroup) per central atom.  The atom's
// neighbour list is staged in LDS sorted by element, as displacement vectors d_ij = R_i - R_j
// (minimum-imaged once when a cell is given) with whatever else of a neighbour the kernel reads
// again (forward and VJP: 16-byte records written by the lane that finds the neighbour; Jacobian:
// one array per quantity); it is either read from a caller-supplied list or built in the kernel
// from the molecule's coordinates with a ballot/popcount compaction (ascending j, same rule as the
// neighbour-list kernel), so the forward/backward pair needs no host round trip for max(nneigh).
//
// Arithmetic per atom (nn neighbours): nn*nRs2 + nn(nn-1)/2*nRs3 exponentials forward;
// the kernels are VALU/transcendental bound, HBM traffic is 4R bytes out (forward) or in
// (VJP) per atom.
//
// The derivatives are written in terms of the three distances a=r_ij, b=r_ik, c=r_jk of a
// triple: every bin value T depends on positions only through (a,b,c) and
// cos_i = (a^2+b^2-c^2)/(2ab) etc., so dT = T_a da + T_b db + T_c dc with
// da/dR_i = u_ij, da/dR_j = -u_ij, db/dR_i = u_ik, db/dR_k = -u_ik, dc/dR_j = u_jk,
// dc/dR_k = -u_jk.  This is algebraically the reference's 40-term expansion; the
// degenerate-angle guard sqrt(max(1e-10, a^2 b^2 - (d_ij.d_ik)^2)) is kept.
#include <algorithm>
#include <type_traits>

#include "qmll_common.h"

namespace {
// 1-ulp forms on the transcendental unit (operands here are distances and widths, far from the
// denormal range): a correctly rounded division, square root or logarithm costs ten or more
// instructions each, several times per neighbour and per triple
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float flog(float x) { return __builtin_amdgcn_logf(x) * 0.6931471805599453f; }
// floor(x / d) for 0 <= x < 1e6, 0 < d: (x + 0.5) / d is at least 0.5 / d away from an integer,
// far more than the rounding of the 1-ulp reciprocal, so the truncation is exact; five
// instructions where the integer division expands to about twenty-five
__device__ __forceinline__ int idiv_small(int x, int d) { return (int)(((float)x + 0.5f) * frcp((float)d)); }

struct FchlArgs {
    const float* X;
    const int* types;
    const float* cell;
    const float* inv_cell;
    const int* atomIDs;
    const int* molIDs;
    const int* natoms;
    const int* nlist;
    const int* nneigh;
    int nn_stride;
    int n;
    int B;
    int cap;  // capacity of the LDS neighbour arrays
    int tcap; // capacity (entries) of the forward kernel's LDS triple table
    const float* Rs2;
    const float* Rs3;
    qmll_fchl_params p;
    float gscale;  // the backward kernel returns gscale * J^T g (folded into the staged gradient row)
};

constexpr int TCH_MAX = 1024;  // longest triple list that the one-wavefront forward kernel is given
constexpr size_t FORWARD_LDS = 5120;   // its LDS request: 32 wavefronts share the 160 KB of a CU
constexpr int TCH_WIDE = 768;  // largest of the several-wavefront one (12 KB): beyond, the triple list is taken in chunks
constexpr int TCH_LEAST = 192; // and its smallest, for capacities that leave no more (up to 1270 neighbours at the default grids)
constexpr float PI_F = 3.14159265358979323846f;
// three floats read from a 16-byte-aligned LDS entry with a single 12-byte instruction (a 16-byte
// read of the same entry occupies the LDS pipe a third longer)
typedef float float3v __attribute__((ext_vector_type(3)));
// an entry of tables that have twelve bytes each, where float3v (sixteen, with a gap) would reach into the next one
struct Float3 {
    float x, y, z;
};
static_assert(sizeof(Float3) == 12, "a table entry");

// LDS neighbour arrays of one central atom, sorted by element type (stable in j within a
// type); goff[e]..goff[e+1] is the slice of type e.
struct Stage {
    float* dx;
    float* dy;
    float* dz;
    float* r;
    float* fc;    // cosine cutoff at r
    float* dfc;   // its r-derivative
    int* el;
    int* j;
    int* goff;    // [ns+1]
    float* next;  // first free float after the neighbour arrays
};

constexpr int STAGE_ARRAYS = 8;   // per-neighbour arrays carved by `carve`

__device__ __forceinline__ Stage carve(float* smem, int cap, int ns) {
    Stage s;
    s.dx = smem;
    s.dy = s.dx + cap;
    s.dz = s.dy + cap;
    s.r = s.dz + cap;
    s.fc = s.r + cap;
    s.dfc = s.fc + cap;
    s.el = (int*)(s.dfc + cap);
    s.j = s.el + cap;
    s.goff = s.j + cap;
    s.next = (float*)(s.goff + ns + 1);
    return s;
}

__device__ __forceinline__ void min_image(float& dx, float& dy, float& dz, const float* c, const float* ic) {
    float s0 = ic[0] * dx + ic[1] * dy + ic[2] * dz;
    float s1 = ic[3] * dx + ic[4] * dy + ic[5] * dz;
    float s2 = ic[6] * dx + ic[7] * dy + ic[8] * dz;
    s0 -= roundf(s0);
    s1 -= roundf(s1);
    s2 -= roundf(s2);
    dx = c[0] * s0 + c[1] * s1 + c[2] * s2;
    dy = c[3] * s0 + c[4] * s1 + c[5] * s2;
    dz = c[6] * s0 + c[7] * s1 + c[8] * s2;
}


// Visit the neighbours of atom (m,i) sorted by element type; returns the neighbour count.
// goff[e]..goff[e+1] becomes the slice of type e, and emit(pos, rank, count, e, j, dx, dy, dz, r2)
// is called once per neighbour by the lane that found it: pos its place in the sorted list, rank
// its place among the `count` neighbours of its type e, j its atom index, d = R_i - R_j.
// Neighbours whose element type is negative (charge not in `species`) are dropped.  Up to 64
// candidates take a single pass; beyond, pass 0 counts per type (lane e keeps the count of type
// e) and pass 1 places each neighbour at goff[type] + its rank among the earlier ones of that type.
template <class Emit>
__device__ __forceinline__ int visit_neighbours(const FchlArgs& a, int* goff, int m, int i, int lane, Emit emit) {
    const float* Xm = a.X + (size_t)m * a.n * 3;
    const int* tm = a.types + (size_t)m * a.n;
    const int ns = a.p.nspecies;
    const bool pbc = a.cell != nullptr;
    float c[9], ic[9];
    if (pbc) {
        for (int t = 0; t < 9; ++t) {
            c[t] = a.cell[(size_t)m * 9 + t];
            ic[t] = a.inv_cell[(size_t)m * 9 + t];
        }
    }
    const float xi = Xm[i * 3 + 0], yi = Xm[i * 3 + 1], zi = Xm[i * 3 + 2];
    // atom `lane` of the molecule, fetched before the atom count is known: without a
    // neighbour list it is this lane's candidate, and the loads overlap the count's
    const int own = lane < a.n ? lane : 0;
    const float xo = Xm[own * 3 + 0], yo = Xm[own * 3 + 1], zo = Xm[own * 3 + 2];
    const int eo = tm[own];
    const float rc2 = a.p.rcut * a.p.rcut;
    const bool have_list = a.nlist != nullptr;
    int total;
    const int* li = nullptr;
    if (have_list) {
        total = a.nneigh[(size_t)m * a.n + i];
        if (total > a.nn_stride) total = a.nn_stride;
        li = a.nlist + ((size_t)m * a.n + i) * a.nn_stride;
    } else {
        total = a.natoms[m];
        if (total > a.n) total = a.n;
    }
    if (total <= QMLL_WAVE) {
        // One candidate per lane: a single pass.  The loads below depend only on the molecule
        // index, so they are issued together; the count of each type is the population of a
        // ballot, known to every lane, and a lane's slot is the running start of its type
        // plus its rank among the earlier lanes of that type.
        const int t = lane;
        const int j = have_list ? (t < total ? li[t] : -1) : t;
        const bool jok = t < total && j >= 0 && j < a.n;
        float xj = xo, yj = yo, zj = zo;
        int e = eo;
        if (have_list) {
            const int jj = jok ? j : 0;
            xj = Xm[jj * 3 + 0];
            yj = Xm[jj * 3 + 1];
            zj = Xm[jj * 3 + 2];
            e = tm[jj];
        }
        float dx = xi - xj, dy = yi - yj, dz = zi - zj;
        if (pbc) min_image(dx, dy, dz, c, ic);
        const float r2 = dx * dx + dy * dy + dz * dz;
        // a supplied list is authoritative (it may be stale on purpose, e.g. finite
        // differences with a frozen list); only the built-in search applies the cutoff
        const bool ok = jok && (have_list ? (r2 > 0.0f) : (r2 < rc2 && r2 > 0.0f)) && e >= 0 && e < ns;
        int start = 0, pos = 0, rank = 0, count = 0;
        const unsigned long long below = (1ull << lane) - 1ull;
        for (int ep = 0; ep < ns; ++ep) {
            const unsigned long long mask = __ballot(ok && e == ep);
            if (lane == 0) goff[ep] = start;
            const int cnt = __popcll(mask);
            if (e == ep) {
                rank = __popcll(mask & below);
                pos = start + rank;
                count = cnt;
            }
            start += cnt;
        }
        const int nn = start < a.cap ? start : a.cap;
        if (lane == 0) goff[ns] = nn;
        if (ok && pos < a.cap) emit(pos, rank, count, e, j, dx, dy, dz, r2);
        return nn;
    }
    int mycount = 0;   // lane e: neighbours of type e seen so far
    int nn = 0;
    for (int pass = 0; pass < 2; ++pass) {
        if (pass == 1) {
            // exclusive prefix over the type counts -> goff
            int incl = mycount;
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(incl, o, 64);
                if (lane >= o) incl += up;
            }
            if (lane < ns) goff[lane] = incl - mycount;
            nn = __shfl(incl, ns - 1, 64);
            if (nn > a.cap) nn = a.cap;
            if (lane == 0) goff[ns] = nn;
            mycount = 0;
            __syncthreads();
        }
        for (int base = 0; base < total; base += QMLL_WAVE) {
            const int t = base + lane;
            bool ok = t < total;
            int j = 0;
            float dx = 0.f, dy = 0.f, dz = 0.f, r2 = 0.f;
            int e = -1;
            if (ok) {
                j = have_list ? li[t] : t;
                ok = j >= 0 && j < a.n;
            }
            if (ok) {
                dx = xi - Xm[j * 3 + 0];
                dy = yi - Xm[j * 3 + 1];
                dz = zi - Xm[j * 3 + 2];
                if (pbc) min_image(dx, dy, dz, c, ic);
                r2 = dx * dx + dy * dy + dz * dz;
                e = tm[j];
                // a supplied list is authoritative (it may be stale on purpose, e.g. finite
                // differences with a frozen list); only the built-in search applies the cutoff
                ok = (have_list ? (r2 > 0.0f) : (r2 < rc2 && r2 > 0.0f)) && e >= 0 && e < ns;
            }
            for (int ep = 0; ep < ns; ++ep) {
                const unsigned long long mask = __ballot(ok && e == ep);
                const int before = __builtin_amdgcn_readlane(mycount, ep);
                if (pass == 1 && ok && e == ep) {
                    const int first = goff[ep];
                    const int rank = before + __popcll(mask & ((1ull << lane) - 1ull));
                    // goff of the last type's end may have been clipped to the capacity
                    if (first + rank < a.cap) emit(first + rank, rank, goff[ep + 1] - first, e, j, dx, dy, dz, r2);
                }
                if (lane == ep) mycount += __popcll(mask);
            }
        }
    }
    return nn;
}

// visit_neighbours for a workgroup of NW wavefronts.  Up to 64 candidates every wavefront does the same single pass
// (equal values go to the same LDS words).  Beyond, each wavefront takes 64 candidates of its own, all loads in
// flight at once, and the places follow from a scan over the (type, wavefront) counts; wcount: NW * nspecies ints of LDS.
// More than 64 NW candidates, or more than 64 / NW types: the two passes of visit_neighbours on every wavefront.
// The caller has a barrier before it reads the list.
template <int NW, class Emit>
__device__ __forceinline__ int visit_neighbours_wide(const FchlArgs& a, int* goff, int* wcount, int m, int i, int tid, Emit emit) {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ns = a.p.nspecies;
    const bool have_list = a.nlist != nullptr;
    int total;
    if (have_list) total = min(a.nneigh[(size_t)m * a.n + i], a.nn_stride);
    else total = min(a.natoms[m], a.n);
    if (total <= QMLL_WAVE || total > QMLL_WAVE * NW || ns * NW > QMLL_WAVE) return visit_neighbours(a, goff, m, i, lane, emit);
    const float* Xm = a.X + (size_t)m * a.n * 3;
    const int* tm = a.types + (size_t)m * a.n;
    int j = tid;
    bool ok = tid < total;
    if (have_list) j = ok ? a.nlist[((size_t)m * a.n + i) * a.nn_stride + tid] : 0;
    ok = ok && j >= 0 && j < a.n;
    const int jj = ok ? j : 0;
    float dx = Xm[i * 3 + 0] - Xm[jj * 3 + 0], dy = Xm[i * 3 + 1] - Xm[jj * 3 + 1], dz = Xm[i * 3 + 2] - Xm[jj * 3 + 2];
    const int e = tm[jj];
    if (a.cell != nullptr) min_image(dx, dy, dz, a.cell + (size_t)m * 9, a.inv_cell + (size_t)m * 9);
    const float r2 = dx * dx + dy * dy + dz * dz;
    ok = ok && (have_list ? r2 > 0.0f : (r2 < a.p.rcut * a.p.rcut && r2 > 0.0f)) && e >= 0 && e < ns;
    int before = 0;                                     // earlier lanes of this wavefront with the same type
    for (int ep = 0; ep < ns; ++ep) {
        const unsigned long long mask = __ballot(ok && e == ep);
        if (e == ep) before = __popcll(mask & ((1ull << lane) - 1ull));
        if (lane == 0) wcount[ep * NW + wave] = __popcll(mask);
    }
    __syncthreads();
    // exclusive scan over the counts, on every wavefront
    const int c = lane < ns * NW ? wcount[lane] : 0;
    int incl = c;
    for (int o = 1; o < ns * NW; o <<= 1) {
        const int up = __shfl_up(incl, o, 64);
        if (lane >= o) incl += up;
    }
    const int excl = incl - c;
    const int nn = min(__shfl(incl, ns * NW - 1, 64), a.cap);
    const int es = ok ? e : 0;
    const int first = __shfl(excl, es * NW, 64);                       // of the type
    const int last = __shfl(incl, es * NW + NW - 1, 64);
    const int pos = __shfl(excl, es * NW + wave, 64) + before;
    if (wave == 0) {
        const int g = __shfl(excl, min(lane * NW, 63), 64);
        if (lane < ns) goff[lane] = g;
        if (lane == 0) goff[ns] = nn;
    }
    if (ok && pos < a.cap) emit(pos, pos - first, last - first, e, j, dx, dy, dz, r2);
    return nn;
}

// the cosine cutoff fc = (cos(pi r / rc) + 1) / 2 and its r-derivative from one sine / cosine pair
__device__ __forceinline__ void cutoff(float r, float inv_rc, float& fc, float& dfc) {
    float sn, cs;
    sincos_hw(r * PI_F * inv_rc, &sn, &cs);
    fc = 0.5f * (cs + 1.0f);
    dfc = -0.5f * PI_F * inv_rc * sn;
}

// the neighbour arrays of `Stage` filled by visit_neighbours
__device__ int stage_neighbours(const FchlArgs& a, const Stage& s, int m, int i, int lane) {
    const float inv_rc = frcp(a.p.rcut);
    return visit_neighbours(a, s.goff, m, i, lane,
                            [&](int pos, int, int, int e, int j, float dx, float dy, float dz, float r2) {
                                const float r = fsqrt(r2);
                                s.dx[pos] = dx;
                                s.dy[pos] = dy;
                                s.dz[pos] = dz;
                                s.r[pos] = r;
                                cutoff(r, inv_rc, s.fc[pos], s.dfc[pos]);
                                s.el[pos] = e;
                                s.j[pos] = j;
                            });
}

// 2^x and log2(x) on the transcendental unit (1 ulp)
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float flog2(float x) { return __builtin_amdgcn_logf(x); }
constexpr float LOG2E = 1.4426950408889634f;

// sqrt(x) from x and its reciprocal root, to half an ulp: sk3 times the last bits of a distance moves the weights of the radial bins
__device__ __forceinline__ float root(float x, float inv) {
    const float r = x * inv;
    return fmaf(0.5f * inv, fmaf(-r, r, x), r);
}

// ---- evenly spaced radial bins --------------------------------------------------------------
// exp2(-(y - u_l)^2) for bins u_l = u_a + k h is w Q^k exp2(-(k h)^2) with w = exp2(-(y - u_a)^2) and Q = exp2(2 h (y - u_a)): the sums over a
// group of five bins are w times a polynomial in Q, whose coefficients take the constant factors, and their derivatives by y follow
// from the polynomial's.  That is one exponential of the transcendental unit per group, and one multiply-add per bin for each sum (Q of all
// groups is one more exponential times a constant each).  Groups of five keep Q^4 in range and its relative error at four
// roundings; where a bin's weight counts, y is near the bin and the arguments of both exponentials are small.  Of 20 bins' 140
// instructions, 20 of them exponentials, 118 and 5 are left.  86016 atoms of 21, three elements, backward 186 -> 172 us; 16 boxes of 96 atoms
// 56.9 -> 50.8, and the forward kernel of several wavefronts per atom, where a lane's second bin is its first times a
// factor of the triple, 48.8 -> 45.8.  The forward kernel of one wavefront per atom keeps both exponentials: the factor
// made its table entries 16 bytes, and 131235 atoms of 3 to 29, five elements went from 275 to 293 us.
constexpr int RS3_GROUP = 5;

// The spacing of the bins u (lane: bin l, if ok) about the middle of the range, to a rounding of the grid's, or 0: uneven, or too wide.
// Q^4 times a coefficient has to be finite, since the weight before it may have underflown.  Where Q could leave 2^(2 line) (y is within mid of the
// middle) or exp2(2 h u) 2^line, `stops` is set, and Q is to stop at 2^24: with bins up to 1.2 apart the weights are below 2^-27 there.  A line
// of 13 leaves room for coefficients of 10^6 and more (20 bins with eta3 = 2.7 up to 8.1 A, 17 up to 7.5); where distances come from a given list and may be
// anything, see group_ratio, it is 8 (6.4 and 5.9 A).  Bins 1.2 apart are those of 12.1 and 10.3 A.
// 42000 atoms of 21, three elements, backward, in groups / one by one: 6 A 78 / 86 us, 8 A 89 / 99, 10 A 90 / 99, 12 A 91 / 100, 17 bins at 6 A 78 / 85; 16 x
// 96 atoms at 8 A 47.1 / 53.2, at 10 A 56.4 / 65.0, at 12 A 62.3 / 70.9.  Errors against 64 bits, 28 and 70 atoms: 6 A 3.5e-7, 8 A 4.1e-7 and 4.5e-7 / 4.3e-7
// and 4.6e-7, 10 A 4.4e-7 and 4.9e-7 / 4.3e-7 and 4.7e-7, 12 A 5.1e-7 and 5.4e-7 / 5.0e-7 and 5.4e-7.
constexpr float LINE_WITHIN = 13.0f, LINE_ANY = 8.0f, WIDEST_SPACING = 1.2f, RATIO_STOP = 16777216.0f;
__device__ __forceinline__ float even_spacing(float u, int l, bool ok, int nRs3, float mid, float line, bool& stops) {
    const float first = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(u)));
    const float last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(u), nRs3 - 1));
    const float h = (last - first) * frcp((float)(nRs3 - 1));
    const float edge = fmaxf(fabsf(first), fabsf(last)), widest = mid + edge;
    const bool fits = fabsf(fmaf((float)-l, h, u - first)) <= 2.4e-7f * widest && fabsf(h) <= WIDEST_SPACING && widest * fabsf(h) <= 40.0f;
    stops = __any(!(widest * fabsf(h) <= line && edge * fabsf(h) <= 0.5f * line));
    return __any(ok && !fits) ? 0.0f : h;
}

// The same for bins 2 l and 2 l + 1 on a lane, l < (nRs3 + 1) / 2 on the first lanes
__device__ __forceinline__ float even_spacing_pairs(float ua, float ub, int l, int nRs3, float mid) {
    const float first = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(ua)));
    const float last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(nRs3 & 1 ? ua : ub), (nRs3 - 1) >> 1));
    const float h = (last - first) * frcp((float)(nRs3 - 1));
    const float edge = fmaxf(fabsf(first), fabsf(last)), widest = mid + edge, slack = 2.4e-7f * widest;
    const float at = fmaf((float)(2 * l), h, first);
    const bool fits = fabsf(ua - at) <= slack && (2 * l + 1 >= nRs3 || fabsf(ub - at - h) <= slack) && widest * fabsf(h) <= LINE_ANY &&
                      edge * fabsf(h) <= 0.5f * LINE_ANY;
    return __any(2 * l < nRs3 && !fits) ? 0.0f : h;
}

// the constant factor of bin l, s = u_l - u_a behind the first of its group: exp2(-s^2), the bin's own place instead of k h where y is on it
__device__ __forceinline__ float group_factor(float u, int l, int lane, float h) {
    const int k = l % RS3_GROUP;
    const float s = u - __shfl(u, lane - k, 64);
    return fexp2(s * (s - 2.0f * h * (float)k));
}

// exp2(2 h y), the factor of Q that all groups share, and what the product's rounding left out: Q goes to the fourth power.
// Distances from a given list may be anything: it stops at 2^STOP (0: not).  2^18 is where the weights are below 2^-49 behind either line (no y of the
// default grid within mid of the middle gets there), and behind LINE_ANY Q^4 stays in range; where Q stops by itself, 2^100.
template <int STOP>
__device__ __forceinline__ float group_ratio(float h, float y) {
    const float x = 2.0f * h * y, e = fexp2(STOP ? fminf(x, (float)STOP) : x);
    return fmaf(e * 0.6931472f, fmaf(2.0f * h, y, -x), e);
}

// G += sum_k g_k w Q^k, H += sum_k g_k (d - k h) w Q^k
__device__ __forceinline__ void group_sums(const float2* g, float d, float w, float Q, float h, float& Gc, float& Gs, float& Hc, float& Hs) {
    const float2 g0 = g[0], g1 = g[1], g2 = g[2], g3 = g[3], g4 = g[4];
    const float hQ = h * Q;
    auto one = [&](float c0, float c1, float c2, float c3, float c4, float& G, float& H) {
        float P = fmaf(c4, Q, c3), D = c4;               // polynomial and derivative
        D = fmaf(D, Q, P);
        P = fmaf(P, Q, c2);
        D = fmaf(D, Q, P);
        P = fmaf(P, Q, c1);
        D = fmaf(D, Q, P);
        P = fmaf(P, Q, c0);
        G = fmaf(w, P, G);
        H = fmaf(w, fmaf(d, P, -hQ * D), H);
    };
    one(g0.x, g1.x, g2.x, g3.x, g4.x, Gc, Hc);
    one(g0.y, g1.y, g2.y, g3.y, g4.y, Gs, Hs);
}

// row index of pair t in the list of pairs (j<k) over nn items, rows enumerated j = 0..nn-2
__device__ __forceinline__ void unrank_pair(int t, int nn, int& j, int& k) {
    const float b = (float)(2 * nn - 1);
    int jj = (int)((b - fsqrt(fmaxf(b * b - 8.0f * (float)t, 0.0f))) * 0.5f);   // first guess; corrected below
    if (jj < 0) jj = 0;
    if (jj > nn - 2) jj = nn - 2;
    // offset(j) = j (2nn - j - 1) / 2
    while (jj > 0 && (jj * (2 * nn - jj - 1)) / 2 > t) --jj;
    while (((jj + 1) * (2 * nn - jj - 2)) / 2 <= t) ++jj;
    j = jj;
    k = jj + 1 + (t - (jj * (2 * nn - jj - 1)) / 2);
}

// pair t of the list of pairs (j<k) enumerated k-major: t = k (k - 1) / 2 + j, 0 <= j < k.  No
// search and no correction step: for t in [k (k - 1) / 2, (k + 1) k / 2) the value 2 t + 1.25 lies in
// [(k - 1/2)^2 + 1, (k + 1/2)^2 - 1], so 1/2 + sqrt(2 t + 1.25) stays at least 1 / (2 k) inside
// (k, k + 1), hundreds of ulps for every t < 2^20 (k < 1449) even with a root two ulps off.
__device__ __forceinline__ void unrank_pair_kmajor(int t, int& j, int& k) {
    k = (int)(0.5f + fsqrt(fmaf(2.0f, (float)t, 1.25f)));
    j = t - (__mul24(k, k - 1) >> 1);
}

__device__ __forceinline__ int pair_offset(int ej, int ek, int ns, int nRs2, int nRs3) {
    const int p = ej < ek ? ej : ek;
    const int q = ej < ek ? ek : ej;
    return ns * nRs2 + 2 * nRs3 * (-(p * (p + 1)) / 2 + q + ns * p);   // fchl_cuda_kernel.cu:658-661
}

// geometry of one triple (central atom i, neighbours j<k in list order)
struct Triple {
    float a, b, c;           // r_ij, r_ik, r_jk
    float ci, cj, ck;        // cosines at i, j, k
    float cosT, sinT;        // cos/sin of the clamped angle at i
    float guard_inv;         // a b / sqrt(max(1e-10, a^2 b^2 - (d_ij.d_ik)^2))
    float ujk[3];            // (R_j - R_k)/c
};

__device__ __forceinline__ Triple triple_geometry(const Stage& s, int j, int k) {
    Triple t;
    const float ax = s.dx[j], ay = s.dy[j], az = s.dz[j];   // d_ij = R_i - R_j
    const float bx = s.dx[k], by = s.dy[k], bz = s.dz[k];   // d_ik
    const float cx = bx - ax, cy = by - ay, cz = bz - az;   // d_jk = R_j - R_k
    t.a = s.r[j];
    t.b = s.r[k];
    const float c2 = cx * cx + cy * cy + cz * cz;
    t.c = fsqrt(c2);
    const float ia = frcp(t.a), ib = frcp(t.b), ic = frcp(t.c);
    const float vi = ax * bx + ay * by + az * bz;           // (R_j-R_i).(R_k-R_i)
    t.ci = vi * ia * ib;
    t.ck = (cx * bx + cy * by + cz * bz) * ic * ib;         // (R_j-R_k).(R_i-R_k)
    t.cj = -(ax * cx + ay * cy + az * cz) * ia * ic;        // (R_i-R_j).(R_k-R_j)
    const float cc = fminf(1.0f, fmaxf(-1.0f, t.ci));
    t.cosT = cc;
    // a^2 b^2 - (d_ij.d_ik)^2 = |d_ij x d_ik|^2 (Lagrange): the cross product keeps full
    // relative accuracy near collinear triples, where the difference of squares cancels
    const float px = ay * bz - az * by, py = az * bx - ax * bz, pz = ax * by - ay * bx;
    const float cross2 = px * px + py * py + pz * pz;
    t.sinT = fminf(1.0f, fsqrt(cross2) * ia * ib);
    t.guard_inv = t.a * t.b * rsqrtf(fmaxf(1e-10f, cross2));
    t.ujk[0] = cx * ic;
    t.ujk[1] = cy * ic;
    t.ujk[2] = cz * ic;
    return t;
}

// what the forward kernels keep of a neighbour, written by the lane that found it: d_ij and 1 / r; sk3 r / 2 - half_mid, fc r^-d3,
// element type, index within the type | neighbours of the type << 16; mu_j, log2(e) / (2 sigma_j^2),
// r^-d2 fc / (sigma sqrt(2 pi))
__device__ __forceinline__ void forward_records(const qmll_fchl_params& p, float sk3, float half_mid, float inv_rc, float* recA, float* recB,
                                                float* s2b, int pos, int rank, int count, int e, float dx, float dy, float dz,
                                                float r2) {
    const float ir = __builtin_amdgcn_rsqf(r2), r = root(r2, ir);
    float fc, dfc;
    cutoff(r, inv_rc, fc, dfc);
    const float l2r = flog2(r);
    const float s2 = flog(fmaf(p.eta2 * ir, ir, 1.0f));
    reinterpret_cast<float4*>(s2b)[pos] = make_float4(
        fmaf(l2r, 0.6931471805599453f, -0.5f * s2),   // ln(r / sqrt(1 + eta2/r^2))
        0.5f * LOG2E * frcp(s2),
        frsq(s2) * 0.3989422804014327f * fexp2(-p.two_body_decay * l2r) * fc, 0.0f);
    reinterpret_cast<float4*>(recA)[pos] = make_float4(dx, dy, dz, ir);
    reinterpret_cast<float4*>(recB)[pos] = make_float4(fmaf(sk3 * 0.5f, r, -half_mid), fc * fexp2(-p.three_body_decay * l2r),
                                                       __int_as_float(e), __int_as_float(rank | (count << 16)));
}

// one table entry per triple: (sk3 rho, K cos, K sin, -) from the two neighbours' records.  With
// a = d_ij, b = d_ik, c = b - a: cos_i cos_j cos_k = -(a.b)(a.c)(c.b) / (|a| |b| |c|)^2, the decay
// (|a| |b| |c|)^-d3 is the product of the neighbours' factors and |c|^-d3 = exp2(-d3 log2(c.c) / 2);
// sin_i = |a x b| / (|a| |b|) keeps full relative accuracy near collinear triples.
__device__ __forceinline__ float4 table_entry(float zw3, float hd3, const float4 Aj, const float4 Bj, const float4 Ak,
                                              const float4 Bk) {
    const float cx = Ak.x - Aj.x, cy = Ak.y - Aj.y, cz = Ak.z - Aj.z;
    const float c2 = cx * cx + cy * cy + cz * cz;
    const float vi = Aj.x * Ak.x + Aj.y * Ak.y + Aj.z * Ak.z;
    const float dac = Aj.x * cx + Aj.y * cy + Aj.z * cz;
    const float dcb = cx * Ak.x + cy * Ak.y + cz * Ak.z;
    const float w = Aj.w * Ak.w;
    const float W = w * frsq(c2);
    const float px = Aj.y * Ak.z - Aj.z * Ak.y, py = Aj.z * Ak.x - Aj.x * Ak.z, pz = Aj.x * Ak.y - Aj.y * Ak.x;
    const float f = zw3 * fmaf(-3.0f * vi * dac, dcb * W * W, 1.0f) * Bj.y * Bk.y * fexp2(hd3 * flog2(c2));
    const float cosT = fminf(1.0f, fmaxf(-1.0f, vi * w));
    const float sinT = fminf(1.0f, fsqrt(px * px + py * py + pz * pz) * w);
    return make_float4(Bj.x + Bk.x, f * cosT, f * sinT, 0.0f);
}

// The triples of an atom as one list ordered by element pair, pairs (p <= q) row by row, each pair's part padded to a multiple
// of `unit` entries: pbase[pq] is its start (written by the wavefront that calls; np + 1 entries).  Returns its length.
// The padding goes to trip[4 t] as zero entries, as far as the list fits tcap of them.
__device__ __forceinline__ int pair_segments(const int* goff, int* pbase, int ns, int np, int lane, int unit, float* trip,
                                             int tcap) {
    int acc = 0;
    for (int q0 = 0; q0 < np; q0 += QMLL_WAVE) {
        int ntr = 0;
        if (q0 + lane < np) {
            int p = 0, rest = q0 + lane;
            while (rest >= ns - p) rest -= ns - p++;
            const int np_ = goff[p + 1] - goff[p], nq = goff[p + rest + 1] - goff[p + rest];
            ntr = rest == 0 ? (__mul24(np_, np_ - 1) >> 1) : __mul24(np_, nq);
        }
        const int size = unit > 1 ? idiv_small(ntr + unit - 1, unit) * unit : ntr;
        int incl = size;
        for (int o = 1; o < QMLL_WAVE && o < np; o <<= 1) {
            const int up = __shfl_up(incl, o, 64);
            if (lane >= o) incl += up;
        }
        if (q0 + lane < np) pbase[q0 + lane + 1] = acc + incl;
        if (q0 == 0 && lane == 0) pbase[0] = 0;
        if (acc + incl <= tcap)
            for (int t = acc + incl - size + ntr; t < acc + incl; ++t)
                reinterpret_cast<float4*>(trip)[t] = make_float4(0.f, 0.f, 0.f, 0.f);
        acc += __shfl(incl, min(63, np - 1 - q0), 64);
    }
    return acc;
}
// where the triple of two neighbours (their second forward records, in list order) stands in the list: k-major within one
// type, row by row else
__device__ __forceinline__ int triple_place(const int* pbase, int ns, const float4 Bj, const float4 Bk) {
    const int p = __float_as_int(Bj.z), q = __float_as_int(Bk.z);   // p <= q: the neighbours are sorted by type
    const int wj = __float_as_int(Bj.w), wk = __float_as_int(Bk.w);
    const int jl = wj & 0xffff, kl = wk & 0xffff;
    return pbase[__mul24(ns, p) - (__mul24(p, p - 1) >> 1) + q - p] +
           (p == q ? (__mul24(kl, kl - 1) >> 1) : __mul24(kl, wj >> 16)) + jl;
}
// and the neighbours of entry tt of the list; false: the entry is padding
__device__ __forceinline__ bool unrank_triple(const int* goff, const int* pbase, int ns, int np, int tt, int& j, int& k) {
    int p = 0, q = 0, pq = 0;
    while (pq + 1 < np && tt >= pbase[pq + 1]) {
        ++pq;
        if (++q == ns) q = ++p;
    }
    const int local = tt - pbase[pq];
    const int nj = goff[p + 1] - goff[p], nk = goff[q + 1] - goff[q];
    bool ok;
    if (p == q) {
        unrank_pair_kmajor(local, j, k);
        ok = k < nj;
    } else {
        k = idiv_small(local, nj);
        j = local - __mul24(k, nj);
        ok = k < nk;
    }
    j += goff[p];
    k += goff[q];
    return ok;
}

// ---------------------------------------------------------------------------------
// forward
//
// Atomic-free: with the neighbours sorted by element type every output block is owned by
// one loop nest.  Two-body block of type e: lanes = (neighbour sub-slot, radial bin z),
// serial over the neighbours of type e, partial sums folded across sub-slots by lane
// shuffles.  Three-body block of the type pair (p<=q): the triples are evaluated
// once (lane = triple) into an LDS table (rho, K cos, K sin) ordered by pair, then lanes = (triple
// sub-slot, radial bin l) run over the pair's part of it with the bin sums in registers.  Rows go
// straight from registers to global memory.  The table holds as many triples as leave room for
// eight wavefronts per SIMD (FORWARD_LDS); a longer list is taken piece by piece.
// ---------------------------------------------------------------------------------
// (96 scalar registers: the eighth wavefront per SIMD; a SIMD has 800 of them, handed out in sixteens, and left
// alone the kernel takes 106.  The thirty-odd values that no longer fit are parked in the lanes of a vector
// register.  The backward kernel's LDS request allows no eighth wavefront, and there the cap only costs.)
__global__ __launch_bounds__(64) __attribute__((amdgpu_num_sgpr(96))) void fchl19_forward_kernel(FchlArgs a,
                                                                                                 float* __restrict__ rep) {
    extern __shared__ float smem[];
    const int lane = threadIdx.x;
    const int m = a.molIDs[blockIdx.x];
    const int i = a.atomIDs[blockIdx.x];
    if (m < 0 || m >= a.B || i < 0 || i >= a.n) return;   // malformed index: write nothing
    const int ns = a.p.nspecies, nRs2 = a.p.nRs2, nRs3 = a.p.nRs3;
    const int R = ns * nRs2 + ns * (ns + 1) * nRs3;

    // LDS: the triple table, three records per neighbour (read with one instruction each), the
    // type offsets, the radial grids, the table's segments
    float* trip = smem;                                  // [tcap][4]: sk3 rho, K cos, K sin, -
    float* recA = trip + 4 * a.tcap;                     // [cap][4]: d_ij, 1 / r
    float* recB = recA + 4 * a.cap;                      // [cap][4]: sk3 r / 2, fc r^-d3, element type,
                                                         //           index within the type | neighbours of the type << 16
    float* s2b = trip;                                   // [cap][4]: mu_j, log2(e) / (2 sigma_j^2), r^-d2 fc / (sigma sqrt(2pi)), -,
                                                         //           done with before the table is filled (tcap >= cap)
    int* goff = (int*)(recB + 4 * a.cap);                // [ns+1] slices of the sorted neighbour list by type
    float* slnRs2 = (float*)(goff + ns + 1);             // [nRs2]
    float* sinvRs2 = slnRs2 + nRs2;                      // [nRs2]
    float* sRs3 = sinvRs2 + nRs2;                        // [nRs3]
    int* pbase = (int*)(sRs3 + nRs3);                    // [np+1] first entry of each element pair in the triple list

    // Global loads that do not depend on the neighbourhood are issued first and consumed after
    // the staging, so their latency overlaps the staging's own loads.
    const float rs2v = lane < nRs2 ? a.Rs2[lane] : 1.0f;
    const float rs3v = lane < nRs3 ? a.Rs3[lane] : 0.0f;
    const float zeta2 = 0.014383766711652736f;   // 2 exp(-pi^2 / 2)
    const float k3 = a.p.eta3 * LOG2E;
    const float sk3 = fsqrt(k3);                 // exp(-eta3 (rho - Rs)^2) = exp2(-(sk3 rho - sk3 Rs)^2)
    const float inv_rc = frcp(a.p.rcut);
    // every neighbour's factors of the two-body bins and of the triples, by the lane that found it
    const int nn = visit_neighbours(
        a, goff, m, i, lane, [&](int pos, int rank, int count, int e, int, float dx, float dy, float dz, float r2) {
            forward_records(a.p, sk3, 0.0f, inv_rc, recA, recB, s2b, pos, rank, count, e, dx, dy, dz, r2);
        });
    if (lane < nRs2) {
        slnRs2[lane] = flog(rs2v);
        sinvRs2[lane] = frcp(rs2v);
    }
    if (lane < nRs3) sRs3[lane] = rs3v;
    for (int t = lane + QMLL_WAVE; t < nRs2; t += QMLL_WAVE) {
        const float v = a.Rs2[t];
        slnRs2[t] = flog(v);
        sinvRs2[t] = frcp(v);
    }
    for (int t = lane + QMLL_WAVE; t < nRs3; t += QMLL_WAVE) sRs3[t] = a.Rs3[t];
    __syncthreads();

    float* out = rep + ((size_t)m * a.n + i) * R;

    // ---- two-body blocks ----
    {
        const int W = nRs2 < 64 ? nRs2 : 64;     // lanes per neighbour sub-slot
        const int JS = idiv_small(64, W);        // neighbour sub-slots
        const int jsub = idiv_small(lane, W), zl = lane - jsub * W;
        for (int zb = 0; zb < nRs2; zb += W) {
            const int z = zb + zl;
            const bool zok = z < nRs2 && jsub < JS;
            const float lnRs = zok ? slnRs2[z] : 0.0f;
            const float invRs = zok ? sinvRs2[z] : 0.0f;
            for (int e = 0; e < ns; ++e) {
                // the same number of rounds for every lane (the loop stays scalar and unrolls);
                // a sub-slot past the end of the type's neighbours reads a valid entry with weight 0
                const int j0 = goff[e], j1 = goff[e + 1];
                const int rounds = idiv_small(j1 - j0 + JS - 1, JS);
                float acc = 0.0f;
#pragma unroll 2
                for (int it = 0; it < rounds; ++it) {
                    const int j = j0 + jsub + it * JS;
                    const bool jok = zok && j < j1;
                    const float3v f = *reinterpret_cast<const float3v*>(s2b + 4 * (jok ? j : j0));   // one 12-byte LDS read
                    const float u = lnRs - f.x;
                    acc = fmaf(jok ? f.z : 0.0f, fexp2(-u * u * f.y), acc);
                }
                acc *= invRs;
                float tot = acc;
                for (int k = 1; k < JS; ++k) tot += __shfl(acc, zl + W * k, 64);
                if (zok && jsub == 0) out[e * nRs2 + z] = tot;
            }
        }
    }

    // ---- three-body blocks ----
    const int W3 = nRs3 < 64 ? nRs3 : 64;
    const int TS = idiv_small(64, W3);
    const int tsub = idiv_small(lane, W3), ll = lane - tsub * W3;
    constexpr int MAXLB = 4;                     // radial bins handled: up to 4 x 64

    const float zw3 = zeta2 * a.p.three_body_weight, hd3 = -0.5f * a.p.three_body_decay;
    const float4* rA = reinterpret_cast<const float4*>(recA);
    const float4* rB = reinterpret_cast<const float4*>(recB);
    // this lane's radial grid points, pre-scaled
    float rsl[MAXLB];
#pragma unroll
    for (int b = 0; b < MAXLB; ++b) {
        const int l = b * 64 + ll;
        rsl[b] = (b * 64 < nRs3) ? sk3 * sRs3[l < nRs3 ? l : 0] : 0.0f;
    }
    const int ntrip = nn * (nn - 1) / 2;
    const int np = ns * (ns + 1) / 2;
    // a pair's part of the list is padded with zero entries to whole rounds, so that every sub-slot runs the same number
    // of rounds and the bin loop is wavefront-uniform (scalar control, unrollable)
    const int length = __builtin_amdgcn_readfirstlane(pair_segments(goff, pbase, ns, np, lane, TS, trip, a.tcap));
    const bool whole = length <= a.tcap;         // the list in one piece, else piece by piece
    __syncthreads();
    // entries t0 .. t1 of the triple list, ordered by element pair, into the table
    auto fill = [&](int t0, int t1) {
        if (whole) {                             // any order of filling does
            for (int tt = lane; tt < ntrip; tt += QMLL_WAVE) {
                int j, k;
                unrank_pair_kmajor(tt, j, k);
                const float4 Aj = rA[j], Ak = rA[k], Bj = rB[j], Bk = rB[k];
                reinterpret_cast<float4*>(trip)[triple_place(pbase, ns, Bj, Bk)] = table_entry(zw3, hd3, Aj, Bj, Ak, Bk);
            }
            return;
        }
        for (int tt = t0 + lane; tt < t1; tt += QMLL_WAVE) {
            int j, k;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (unrank_triple(goff, pbase, ns, np, tt, j, k)) v = table_entry(zw3, hd3, rA[j], rB[j], rA[k], rB[k]);
            reinterpret_cast<float4*>(trip)[tt - t0] = v;
        }
    };
    float* out3 = out + ns * nRs2;               // the pairs' blocks follow each other in list order

    // The rest of the kernel, with the sub-slot count as a compile-time constant where it is one of
    // the common ones (TSC = 0: any): the table reads of a round then sit at fixed offsets from
    // one address per lane.
    auto three_body = [&](auto tsc) {
        constexpr int TSC = decltype(tsc)::value;
        const int TSv = TSC ? TSC : TS;
        const int tsafe = tsub < TSv ? tsub : 0;
        // bin sums of `rounds` rounds of table entries starting at `from`, added to the accumulators
        auto accumulate = [&](int from, int rounds, float (&accc)[MAXLB], float (&accs)[MAXLB]) {
            const float4* src = reinterpret_cast<const float4*>(trip) + from + tsafe;
#pragma unroll
            for (int b = 0; b < MAXLB; ++b) {
                if (b * 64 < nRs3) {
                    const float rs = rsl[b];
                    float c_ = accc[b], s_ = accs[b];
#pragma unroll 4
                    for (int it = 0; it < rounds; ++it) {
                        const float3v v = *reinterpret_cast<const float3v*>(src + it * TSv);   // one 12-byte LDS read
                        const float d = v.x - rs;
                        const float e = fexp2(-d * d);
                        c_ = fmaf(e, v.y, c_);
                        s_ = fmaf(e, v.z, s_);
                    }
                    accc[b] = c_;
                    accs[b] = s_;
                }
            }
        };
        // fold the triple sub-slots and store the pair's block
        auto store_block = [&](int pq, bool any, const float (&accc)[MAXLB], const float (&accs)[MAXLB]) {
#pragma unroll
            for (int b = 0; b < MAXLB; ++b) {
                if (b * 64 < nRs3) {
                    float tc = accc[b], tsn = accs[b];
                    if (any) {
                        for (int k = 1; k < TSv; ++k) {
                            tc += __shfl(accc[b], ll + W3 * k, 64);
                            tsn += __shfl(accs[b], ll + W3 * k, 64);
                        }
                    }
                    const int l = b * 64 + ll;
                    if (tsub == 0 && l < nRs3) {
                        const float2 v = make_float2(tc, tsn);
                        __builtin_memcpy(out3 + 2 * (pq * nRs3 + l), &v, sizeof v);   // one 8-byte store, 4-byte aligned
                    }
                }
            }
        };
        int first = 0, last = min(a.tcap, length);                   // what the table holds
        fill(first, last);
        __syncthreads();
        int pos = 0;
        for (int pq = 0; pq < np; ++pq) {
            const int begin = pos, end = __builtin_amdgcn_readfirstlane(pbase[pq + 1]);
            float accc[MAXLB], accs[MAXLB];
#pragma unroll
            for (int b = 0; b < MAXLB; ++b) accc[b] = accs[b] = 0.0f;
            if (__builtin_expect(end > last, 0)) {
                // the pair's part goes beyond the table: refill until its last piece is there
                do {
                    accumulate(pos - first, idiv_small(last - pos, TSv), accc, accs);
                    pos = first = last;
                    last = min(first + a.tcap, length);
                    __syncthreads();
                    fill(first, last);
                    __syncthreads();
                } while (end > last);
            }
            const bool any = end > begin;        // the elements of the pair are both there
            if (any) accumulate(pos - first, idiv_small(end - pos, TSv), accc, accs);
            pos = end;
            store_block(pq, any, accc, accs);
        }
    };
    switch (TS) {
        case 1: three_body(std::integral_constant<int, 1>{}); break;
        case 2: three_body(std::integral_constant<int, 2>{}); break;
        case 3: three_body(std::integral_constant<int, 3>{}); break;
        case 4: three_body(std::integral_constant<int, 4>{}); break;
        default: three_body(std::integral_constant<int, 0>{}); break;
    }
}

// ---------------------------------------------------------------------------------
// forward, one wavefront per central atom, number of elements known to the compiler
//
// The same sums as fchl19_forward_kernel for the usual grids (LEAN_RS3 - 3 .. LEAN_RS3 three-body and up to 32 two-body bins), up to
// five elements, no given list and at most 64 candidates, which one instruction's lanes hold.  That kernel is bound by the number of
// its instructions, vector, scalar and LDS ones alike (1121 + 615 + 126 per atom of 20 neighbours and three elements), and by the LDS:
// its bin loop reads 12 bytes per lane for one exponential, and the four SIMDs share 128 bytes a clock.  Here
//  * the counts of the elements are scalars, so that the pairs' segments need no scan and no LDS, and all loops over elements and
//    pairs are unrolled;
//  * a lane holds two radial bins (six triples at a time instead of three), so that one read serves two exponentials, and the sums
//    of six pairs are exchanged at once: 20 shuffles and one store instead of 24 and six;
//  * a neighbour's record says where each of its triples stands, and a table entry has 12 bytes instead of 16, so that the whole
//    list of 29 atoms fits 6.5 KB (a list in pieces costs a search per triple).
// 967 + 251 + 122 instructions; 86016 atoms of 21, three elements 186 -> 136 us, 131235 atoms of 3 to 29, five elements 337 -> 251,
// 64000 of 8 82 -> 50, 80000 of 40 413 -> 354.  Vector issue now takes nine tenths of the launch.  Two, four or eight atoms per
// workgroup (fewer dispatches) and other depths of unrolling made no difference.
// ---------------------------------------------------------------------------------
constexpr int LEAN_RS3 = 20, LEAN_SLOTS = 6, LEAN_LANES = 10;    // bins; triples at a time, lanes (two bins each) of each
// What qmll_prepare_batch does for a small batch, by workgroups of the forward launch beside those of the atoms
struct BatchPrep {
    const float* Z;              // null: done by a launch of its own
    const float* species;
    const float* model_species;  // null: the model goes by `species`
    int ne;                      // elements of the model
    int A;
    int slots;
    int* types;
    int* sort_types;
    int* sorted;
    int* offsets;
    float* zero;
    int zero_count;
    int groups;                  // workgroups: the sort, then 256 slots and floats each
};
constexpr int PREP_ATOMS = 256, PREP_ELEMENTS = 8;

// group 0: the listed atoms sorted by the model's element (stable), one wavefront, 64 atoms at a time; the others: element indices of
// the slots (0 for padded ones) and the zeros
__device__ __forceinline__ void prepare_group(const FchlArgs& a, const BatchPrep& b, int group, int lane, int* lds) {
    const float* list = b.model_species ? b.model_species : b.species;
    const int ns = a.p.nspecies, nlist = b.model_species ? b.ne : ns;
    if (group > 0) {
        const int step = 64 * (b.groups - 1);
        for (int s = (group - 1) * 64 + lane; s < b.slots; s += step) {
            const int m = s / a.n;
            const bool real = s - m * a.n < a.natoms[m];
            b.types[s] = real ? species_index(b.Z[s], b.species, ns) : 0;
            if (b.model_species) b.sort_types[s] = real ? species_index(b.Z[s], b.model_species, b.ne) : 0;
        }
        for (int t = (group - 1) * 64 + lane; t < b.zero_count; t += step) b.zero[t] = 0.0f;
        return;
    }
    int total[PREP_ELEMENTS];
#pragma unroll
    for (int e = 0; e < PREP_ELEMENTS; ++e) total[e] = 0;
#pragma unroll
    for (int base = 0; base < PREP_ATOMS; base += QMLL_WAVE) {         // all loads in flight
        const int at = base + lane;
        int slot = 0, t = -1;
        if (at < b.A) {
            const int m = a.molIDs[at], i = a.atomIDs[at];
            slot = m * a.n + i;
            t = i < a.natoms[m] ? species_index(b.Z[slot], list, nlist) : 0;
            lds[at] = slot << 4 | (t + 1);
        }
#pragma unroll
        for (int e = 0; e < PREP_ELEMENTS; ++e) total[e] += __popcll(__ballot(t == e));
    }
    int start = 0;
#pragma unroll
    for (int e = 0; e < PREP_ELEMENTS; ++e) {
        const int n = total[e];
        total[e] = start;                                // from here: where the next of this element goes
        if (lane == 0 && e <= b.ne) b.offsets[e] = start;
        start += n;
    }
    if (lane == 0 && b.ne == PREP_ELEMENTS) b.offsets[b.ne] = start;
    for (int base = 0; base < b.A; base += QMLL_WAVE) {
        const int at = base + lane;
        const int v = at < b.A ? lds[at] : 0;
        const int t = (v & 15) - 1;
#pragma unroll
        for (int e = 0; e < PREP_ELEMENTS; ++e) {
            const unsigned long long mask = __ballot(t == e);
            if (t == e) b.sorted[total[e] + __popcll(mask & ((1ull << lane) - 1ull))] = v >> 4;
            total[e] += __popcll(mask);
        }
    }
    // entries past the last typed atom name a valid slot, so gathers through them stay in bounds
    for (int k = start + lane; k < b.A; k += QMLL_WAVE) b.sorted[k] = 0;
}

// what a wavefront wrote to LDS is there for its own lanes: LDS takes a wavefront's instructions in order
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One wavefront writes atom i's row to `out`; FROM_CHARGES: the elements are taken from the charges.  sync: what makes the wavefront's LDS writes
// visible to itself.
template <int NS, bool FROM_CHARGES, class Sync>
__device__ __forceinline__ void lean_forward(const FchlArgs& a, const BatchPrep& b, int m, int i, int lane, float* smem, float* out, Sync sync) {
    constexpr int NP = NS * (NS + 1) / 2;
    const int nRs2 = a.p.nRs2, nRs3 = a.p.nRs3;
    float* recA = smem;                                  // [cap][4]: d_ij, 1 / r
    float* recB = recA + 4 * a.cap;                      // [cap][4]: sk3 r / 2, fc r^-d3, places (below)
    float* trip = recB + 4 * a.cap;                      // [tcap][3]: sk3 rho, K cos, K sin; before them the two-body factors [cap][3]

    const float* Xm = a.X + (size_t)m * a.n * 3;
    const int own = lane < a.n ? lane : 0;
    const float xj = Xm[own * 3 + 0], yj = Xm[own * 3 + 1], zj = Xm[own * 3 + 2];
    const int et = FROM_CHARGES ? species_index(b.Z[(size_t)m * a.n + own], b.species, NS) : a.types[(size_t)m * a.n + own];
    const int z = lane & 31, half = lane >> 5;           // two-body: radial bin, neighbour of two
    const float rs2v = z < nRs2 ? a.Rs2[z] : 1.0f;
    const int slot = idiv_small(lane, LEAN_LANES), ll = lane - LEAN_LANES * slot;      // three-body: triple of six, pair of bins
    const float rs3a = 2 * ll < nRs3 ? a.Rs3[2 * ll] : 0.0f, rs3b = 2 * ll + 1 < nRs3 ? a.Rs3[2 * ll + 1] : 0.0f;
    const int total = min(a.natoms[m], a.n);

    const float zeta2 = 0.014383766711652736f;   // 2 exp(-pi^2 / 2)
    const float sk3 = fsqrt(a.p.eta3 * LOG2E);   // exp(-eta3 (rho - Rs)^2) = exp2(-(sk3 rho - sk3 Rs)^2)
    const float inv_rc = frcp(a.p.rcut);

    // ---- neighbours: candidate = lane ----
    float dx = Xm[i * 3 + 0] - xj, dy = Xm[i * 3 + 1] - yj, dz = Xm[i * 3 + 2] - zj;
    if (a.cell != nullptr) min_image(dx, dy, dz, a.cell + (size_t)m * 9, a.inv_cell + (size_t)m * 9);
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool near = lane < total && r2 < a.p.rcut * a.p.rcut && r2 > 0.0f;
    int count[NS], first[NS], rounds[NP], base[NP];
    const unsigned long long below = (1ull << lane) - 1ull;
    int rank = 0, nn = 0;
#pragma unroll
    for (int e = 0; e < NS; ++e) {
        const unsigned long long mask = __ballot(near && et == e);
        count[e] = __popcll(mask);
        first[e] = nn;
        nn += count[e];
        if (et == e) rank = __popcll(mask & below);
    }
    // the triples of an element pair are consecutive in the table, pairs row by row, each part padded to whole rounds
    int length = 0;
#pragma unroll
    for (int p = 0, pq = 0; p < NS; ++p)
#pragma unroll
        for (int q = p; q < NS; ++q, ++pq) {
            const int n = p == q ? (count[p] * (count[p] - 1)) >> 1 : count[p] * count[q];
            rounds[pq] = (unsigned)(n + LEAN_SLOTS - 1) / LEAN_SLOTS;
            base[pq] = length;
            length += LEAN_SLOTS * rounds[pq];
        }
    if (near && et >= 0 && et < NS) {
        // Where a triple of neighbours j < k (in list order) stands: place[type of j] + j, from k's record.  Five places of 11 bits
        // and, above them, 11 times k's own type.  (A place is not negative: with type p there, the parts before (p, q) hold
        // at least one triple for each neighbour of an earlier type.)
        unsigned lo = 0, hi = 0;
        int pos = rank;
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            if (et == q) {
                unsigned t[5] = {0, 0, 0, 0, 0};
#pragma unroll
                for (int p = 0; p <= q; ++p) {
                    const int pq = p * NS - p * (p - 1) / 2 + q - p;
                    t[p] = (unsigned)(base[pq] - first[p] + (p == q ? __mul24(rank, rank - 1) >> 1 : __mul24(rank, count[p]))) & 0x7ff;
                }
                lo = t[0] | t[1] << 11 | t[2] << 22;
                hi = t[2] >> 10 | t[3] << 1 | t[4] << 12 | (unsigned)(11 * q) << 23;
                pos = rank + first[q];
            }
        }
        const float ir = __builtin_amdgcn_rsqf(r2), r = root(r2, ir);
        float fc, dfc;
        cutoff(r, inv_rc, fc, dfc);
        const float l2r = flog2(r);
        const float s2 = flog(fmaf(a.p.eta2 * ir, ir, 1.0f));
        reinterpret_cast<float4*>(recA)[pos] = make_float4(dx, dy, dz, ir);
        reinterpret_cast<float4*>(recB)[pos] = make_float4(sk3 * 0.5f * r, fc * fexp2(-a.p.three_body_decay * l2r),
                                                           __uint_as_float(lo), __uint_as_float(hi));
        float* f2 = trip + 3 * pos;                       // mu, log2(e) / (2 sigma^2), r^-d2 fc / (sigma sqrt(2 pi))
        f2[0] = fmaf(l2r, 0.6931471805599453f, -0.5f * s2);
        f2[1] = 0.5f * LOG2E * frcp(s2);
        f2[2] = frsq(s2) * 0.3989422804014327f * fexp2(-a.p.two_body_decay * l2r) * fc;
    }
    sync();

    // ---- two-body blocks ----
    {
        const float lnRs = flog(rs2v), invRs = frcp(rs2v);
#pragma unroll
        for (int e = 0; e < NS; ++e) {
            const float* f = trip + 3 * (first[e] + half);
            float acc = 0.0f;
            auto add = [&](const float* at, bool there) {
                Float3 v;
                __builtin_memcpy(&v, at, sizeof v);
                const float u = lnRs - v.x;
                acc = fmaf(there ? v.z : 0.0f, fexp2(-u * u * v.y), acc);
            };
            const int twos = count[e] >> 1;
#pragma unroll 2
            for (int it = 0; it < twos; ++it, f += 6) add(f, true);
            if (count[e] & 1) add(half ? f - 3 : f, half == 0);
            acc *= invRs;
            acc += lane_xor<32>(acc);
            if (lane < nRs2) out[e * nRs2 + lane] = acc;
        }
    }
    sync();

    // ---- the table ----
    {
        const float zw3 = zeta2 * a.p.three_body_weight, hd3 = -0.5f * a.p.three_body_decay;
        const float4* rA = reinterpret_cast<const float4*>(recA);
        const float4* rB = reinterpret_cast<const float4*>(recB);
        for (int t = lane; 4 * t < 3 * length; t += QMLL_WAVE)               // the padding
            reinterpret_cast<float4*>(trip)[t] = make_float4(0.f, 0.f, 0.f, 0.f);
        const int ntrip = (nn * (nn - 1)) >> 1;
        for (int tt = lane; tt < ntrip; tt += QMLL_WAVE) {
            int j, k;
            unrank_pair_kmajor(tt, j, k);
            const float4 Aj = rA[j], Ak = rA[k], Bj = rB[j], Bk = rB[k];
            const unsigned long long places = (unsigned long long)__float_as_uint(Bk.w) << 32 | __float_as_uint(Bk.z);
            const int at = (int)((unsigned)(places >> (__float_as_uint(Bj.w) >> 23)) & 0x7ff) + j;
            const float4 v = table_entry(zw3, hd3, Aj, Bj, Ak, Bk);
            const Float3 w = {v.x, v.y, v.z};
            __builtin_memcpy(trip + 3 * at, &w, sizeof w);
        }
    }
    sync();

    // ---- three-body blocks ----
    const float rsa = sk3 * rs3a, rsb = sk3 * rs3b;
    const float* src = trip + (slot < LEAN_SLOTS ? 3 * slot : 0);
    float* out3 = out + NS * nRs2;
#pragma unroll
    for (int g = 0; g < NP; g += LEAN_SLOTS) {
        float v[LEAN_SLOTS][4];
#pragma unroll
        for (int s = 0; s < LEAN_SLOTS; ++s) {
            float c0 = 0.f, s0 = 0.f, c1 = 0.f, s1 = 0.f;
            if (g + s < NP) {
#pragma unroll 2
                for (int it = 0; it < rounds[g + s < NP ? g + s : 0]; ++it, src += 3 * LEAN_SLOTS) {
                    Float3 t;
                    __builtin_memcpy(&t, src, sizeof t);
                    const float d0 = t.x - rsa, d1 = t.x - rsb;
                    const float e0 = fexp2(-d0 * d0), e1 = fexp2(-d1 * d1);
                    c0 = fmaf(e0, t.y, c0);
                    s0 = fmaf(e0, t.z, s0);
                    c1 = fmaf(e1, t.y, c1);
                    s1 = fmaf(e1, t.z, s1);
                }
            }
            v[s][0] = c0, v[s][1] = s0, v[s][2] = c1, v[s][3] = s1;
        }
        // the six slots' sums of six element pairs: slot s ends up with pair s.  First between slots s and s + 3, each of which keeps
        // three of the pairs, then among the three slots that hold the same three
        float w[3][4];
        const bool upper = slot >= 3;
        const int other = upper ? lane - 30 : lane + 30;
#pragma unroll
        for (int s = 0; s < 3; ++s)
#pragma unroll
            for (int c = 0; c < 4; ++c) w[s][c] = (upper ? v[s + 3][c] : v[s][c]) + __shfl(upper ? v[s][c] : v[s + 3][c], other, 64);
        const int h = upper ? slot - 3 : slot;
        const int next = h == 2 ? lane - 20 : lane + 10, last = h == 0 ? lane + 20 : lane - 10;
        float4 o;
        float* po = &o.x;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float mine = h == 0 ? w[0][c] : h == 1 ? w[1][c] : w[2][c];
            const float from_next = __shfl(h == 0 ? w[2][c] : h == 1 ? w[0][c] : w[1][c], next, 64);    // the slot after this one: what it holds of mine
            const float from_last = __shfl(h == 0 ? w[1][c] : h == 1 ? w[2][c] : w[0][c], last, 64);
            po[c] = mine + from_next + from_last;
        }
        if (slot < LEAN_SLOTS && g + slot < NP) {
            float* to = out3 + 2 * ((g + slot) * nRs3 + 2 * ll);
            if (2 * ll + 1 < nRs3) __builtin_memcpy(to, &o, 16);
            else if (2 * ll < nRs3) __builtin_memcpy(to, &o, 8);
        }
    }
}

// PREP: the first groups of the launch prepare the batch, the atoms' workgroups take the elements from the charges (no launch ahead of
// this one has written the types).
template <int NS, bool PREP>
__global__ __launch_bounds__(64) void fchl19_forward_lean_kernel(FchlArgs a, BatchPrep b, float* __restrict__ rep) {
    extern __shared__ float smem[];
    const int lane = threadIdx.x;
    int atom = blockIdx.x;
    if constexpr (PREP) {
        if (atom < b.groups) {
            prepare_group(a, b, atom, lane, reinterpret_cast<int*>(smem));
            return;
        }
        atom -= b.groups;
    }
    const int m = a.molIDs[atom];
    const int i = a.atomIDs[atom];
    if (m < 0 || m >= a.B || i < 0 || i >= a.n) return;   // malformed index: write nothing
    const int R = NS * a.p.nRs2 + NS * (NS + 1) * a.p.nRs3;
    lean_forward<NS, PREP>(a, b, m, i, lane, smem, rep + ((size_t)m * a.n + i) * R, [] { __syncthreads(); });
}

// The representation of few atoms and its projection in one launch, beside the preparation of the batch: a workgroup per atom, whose first
// wavefront forms the row in LDS while the reductor's rows are on their way into the registers of all eight and the others count
// the atom's place in the sorted list.  x[place, :] = row . U.  21 atoms of three elements, 128 components: 6.5 + 4.3 us in two launches, 9.6 so,
// and 4 us of the host's time for the launch.
// PREP = false: the batch has been prepared, and the workgroups follow the sorted list.
constexpr int MOST_WAVES = 8;
// rows of a reductor that the registers of eight wavefronts hold beside the rest, in both directions: five elements of the default grids at
// 64 components, four at 128; of four and two wavefronts
constexpr int held_rows(int d, int waves) { return waves == MOST_WAVES ? (d == 64 ? 768 : 512) : 96 * waves * 64 / d; }
constexpr int fewest_rows(int ns) { return ns + ns * (ns + 1) * (LEAN_RS3 - 3); }                // that a representation of the lean grids has
template <int NS, int D, int W, bool PREP>
__global__ __launch_bounds__(64 * W) void fchl19_forward_projected_kernel(FchlArgs a, BatchPrep b, const float* __restrict__ reductors,
                                                                          float* __restrict__ x) {
    static_assert(!PREP || W > PREP_ATOMS / 64, "a wavefront for every 64 atoms of the list, and one for the representation");
    extern __shared__ float smem[];
    constexpr int CL = D / 4, KS = 64 * W / CL, MINE = held_rows(D, W) / KS;     // lanes along the columns, slices of the rows, rows of each
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (PREP && (int)blockIdx.x < b.groups) {
        if (wave == 0) prepare_group(a, b, blockIdx.x, lane, reinterpret_cast<int*>(smem));
        return;
    }
    const int atom = PREP ? blockIdx.x - b.groups : blockIdx.x, R = NS * a.p.nRs2 + NS * (NS + 1) * a.p.nRs3;
    const float* list = b.model_species ? b.model_species : b.species;
    const int nlist = b.model_species ? b.ne : a.p.nspecies;
    // element of a listed atom by the model's list, as prepare_group has it; -1: not in the sorted list
    auto element = [&](int at) {
        const int m = a.molIDs[at], i = a.atomIDs[at];
        if (m < 0 || m >= a.B || i < 0 || i >= a.n) return -1;
        return i < a.natoms[m] ? species_index(b.Z[(size_t)m * a.n + i], list, nlist) : 0;
    };
    int m, i, e = 0;
    if constexpr (PREP) {
        m = a.molIDs[atom];
        i = a.atomIDs[atom];
        e = __builtin_amdgcn_readfirstlane(element(atom));
    } else {
        if (atom >= b.offsets[b.ne]) return;
        while (e + 1 < b.ne && atom >= b.offsets[e + 1]) ++e;
        const int slot = b.sorted[atom];
        m = slot / a.n;
        i = slot - m * a.n;
    }
    if (m < 0 || m >= a.B || i < 0 || i >= a.n || e < 0 || e >= b.ne) return;
    float* row = smem;                                   // [R4] the representation
    float* part = row + ((R + 3) & ~3);                  // [W][D]
    int* before = reinterpret_cast<int*>(part + W * D);  // [PREP_ATOMS / 64]
    float* own = reinterpret_cast<float*>(before + PREP_ATOMS / 64);
    const int c4 = tid % CL, ks = tid / CL;
    const float4* U = reinterpret_cast<const float4*>(reductors + (size_t)e * R * D) + c4;
    float4 u[MINE];
#pragma unroll
    for (int k = 0; k < MINE; ++k) {
        u[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (KS * k < R) u[k] = U[(size_t)min(ks + KS * k, R - 1) * CL];
    }
    if (wave == 0) {
        lean_forward<NS, PREP>(a, b, m, i, lane, own, row, [] { wave_sync(); });
    } else if (PREP && wave <= PREP_ATOMS / 64) {                // the atoms ahead of this one in the sorted list
        const int at = tid - 64;
        const int t = at < b.A ? element(at) : -1;
        const int count = __popcll(__ballot(t >= 0 && (t < e || (t == e && at < atom))));
        if (lane == 0) before[wave - 1] = count;
    }
    __syncthreads();
    float4 sums[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
#pragma unroll
    for (int k = 0; k < MINE; ++k) {
        if (KS * k >= R) break;
        const float r = ks + KS * k < R ? row[ks + KS * k] : 0.0f;
        float4& t = sums[k & 1];
        t.x = fmaf(r, u[k].x, t.x);
        t.y = fmaf(r, u[k].y, t.y);
        t.z = fmaf(r, u[k].z, t.z);
        t.w = fmaf(r, u[k].w, t.w);
    }
    float4 acc = make_float4(sums[0].x + sums[1].x, sums[0].y + sums[1].y, sums[0].z + sums[1].z, sums[0].w + sums[1].w);
    float* v = &acc.x;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if constexpr (CL == 16) v[c] += lane_xor<16>(v[c]);
        v[c] += lane_xor<32>(v[c]);
    }
    if (lane < CL) reinterpret_cast<float4*>(part)[wave * CL + lane] = acc;
    __syncthreads();
    if (tid < D) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) sum += part[w * D + tid];
        int place = PREP ? 0 : atom;
        if constexpr (PREP) {
#pragma unroll
            for (int w = 0; w < PREP_ATOMS / 64; ++w) place += before[w];
        }
        x[(size_t)place * D + tid] = sum;
    }
}

// ---------------------------------------------------------------------------------
// forward, several wavefronts per central atom
//
// For neighbourhoods too large for one wavefront's table (beyond 46 atoms) and for batches of few atoms, where one
// wavefront per atom leaves the chip idle and the launch takes as long as one atom's chain of phases.  The
// triple list, ordered by element pair, is taken in chunks of the table (one chunk where it fits): all wavefronts fill
// the table, each sums a run of its entries, and the NW partial blocks are added
// in a fixed order at the end: deterministic like the kernel above.
// ---------------------------------------------------------------------------------
template <int NW, bool LEAN>
__global__ __launch_bounds__(64 * NW) void fchl19_forward_wide_kernel(FchlArgs a, float* __restrict__ rep) {
    extern __shared__ float smem[];
    constexpr int NT = 64 * NW;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = a.molIDs[blockIdx.x];
    const int i = a.atomIDs[blockIdx.x];
    if (m < 0 || m >= a.B || i < 0 || i >= a.n) return;   // malformed index: write nothing
    const int ns = a.p.nspecies, nRs2 = a.p.nRs2, nRs3 = a.p.nRs3;
    const int np = ns * (ns + 1) / 2;
    const int R = ns * nRs2 + 2 * np * nRs3;

    const int per = 2 * nRs3;
    float* trip = smem;                                  // [tcap + 1][4], the last entry zero
    float* recA = trip + 4 * (a.tcap + 1);
    float* recB = recA + 4 * a.cap;
    float* s2b = recB + 4 * a.cap;
    // [np][NW][2 nRs3] partial blocks; one wavefront adds into the row itself
    float* part = NW > 1 ? s2b + 4 * a.cap : rep + ((size_t)m * a.n + i) * R + ns * nRs2;
    int* goff = (int*)(s2b + 4 * a.cap + (NW > 1 ? (size_t)np * NW * per : 0));
    float* slnRs2 = (float*)(goff + ns + 1);
    float* sinvRs2 = slnRs2 + nRs2;
    float* sRs3 = sinvRs2 + nRs2;
    int* pbase = (int*)(sRs3 + nRs3);                    // [np + 1] first entry of each pair in the triple list
    int* wcount = pbase + np + 1;                        // [ns * NW]

    const float zeta2 = 0.014383766711652736f;   // 2 exp(-pi^2 / 2)
    const float sk3 = fsqrt(a.p.eta3 * LOG2E);
    const float inv_rc = frcp(a.p.rcut);
    const float mid = LEAN ? 0.5f * sk3 * a.p.rcut : 0.0f;       // LEAN: distances and bins about the middle of the range
    const float rs2v = tid < nRs2 ? a.Rs2[tid] : 1.0f;
    const float rs3v = tid < nRs3 ? a.Rs3[tid] : 0.0f;
    const int nn = visit_neighbours_wide<NW>(
        a, goff, wcount, m, i, tid, [&](int pos, int rank, int count, int e, int, float dx, float dy, float dz, float r2) {
            forward_records(a.p, sk3, 0.5f * mid, inv_rc, recA, recB, s2b, pos, rank, count, e, dx, dy, dz, r2);
        });
    for (int t = tid; t < np * NW * per; t += NT) part[t] = 0.0f;
    for (int t = tid; t < nRs2; t += NT) {
        const float v = t == tid ? rs2v : a.Rs2[t];
        slnRs2[t] = flog(v);
        sinvRs2[t] = frcp(v);
    }
    for (int t = tid; t < nRs3; t += NT) sRs3[t] = t == tid ? rs3v : a.Rs3[t];
    if (tid < 4) trip[4 * a.tcap + tid] = 0.0f;
    __syncthreads();

    float* out = rep + ((size_t)m * a.n + i) * R;

    // two-body blocks: an element type per wavefront
    {
        const int W = nRs2 < 64 ? nRs2 : 64;
        const int JS = idiv_small(64, W);
        const int jsub = idiv_small(lane, W), zl = lane - jsub * W;
        for (int e = wave; e < ns; e += NW) {
            const int j0 = goff[e], j1 = goff[e + 1];
            const int rounds = idiv_small(j1 - j0 + JS - 1, JS);
            for (int zb = 0; zb < nRs2; zb += W) {
                const int z = zb + zl;
                const bool zok = z < nRs2 && jsub < JS;
                const float lnRs = zok ? slnRs2[z] : 0.0f;
                const float invRs = zok ? sinvRs2[z] : 0.0f;
                float acc = 0.0f;
#pragma unroll 2
                for (int it = 0; it < rounds; ++it) {
                    const int j = j0 + jsub + it * JS;
                    const bool jok = zok && j < j1;
                    const float3v f = *reinterpret_cast<const float3v*>(s2b + 4 * (jok ? j : j0));
                    const float u = lnRs - f.x;
                    acc = fmaf(jok ? f.z : 0.0f, fexp2(-u * u * f.y), acc);
                }
                acc *= invRs;
                float tot = acc;
                for (int k = 1; k < JS; ++k) tot += __shfl(acc, zl + W * k, 64);
                if (zok && jsub == 0) out[e * nRs2 + z] = tot;
            }
        }
    }
    pair_segments(goff, pbase, ns, np, lane, 1, trip, 0);   // the same on every wavefront
    __syncthreads();

    const int W3 = LEAN ? LEAN_LANES : nRs3 < 64 ? nRs3 : 64;      // LEAN: two bins per lane, see fchl19_forward_lean_kernel
    const int TS = LEAN ? LEAN_SLOTS : idiv_small(64, W3);
    const int tsub = idiv_small(lane, W3), ll = lane - tsub * W3;
    constexpr int MAXLB = 4;                             // radial bins handled: up to 4 x 64
    float rsl[MAXLB];
#pragma unroll
    for (int b = 0; b < (LEAN ? 2 : MAXLB); ++b) {
        const int l = LEAN ? 2 * ll + b : b * 64 + ll;
        rsl[b] = (LEAN || b * 64 < nRs3) ? fmaf(sk3, sRs3[l < nRs3 ? l : 0], -mid) : 0.0f;
    }
    // LEAN, an even grid: the second of a lane's two weights is the first times exp2(2 h y), once per triple, and this constant
    const float h = LEAN ? even_spacing_pairs(rsl[0], rsl[1], ll, nRs3, mid) : 0.0f;
    const float step = rsl[1] - rsl[0], factor = LEAN && h != 0.0f ? fexp2(step * (step - 2.0f * h) - 2.0f * h * rsl[0]) : 1.0f;
    const float zw3 = zeta2 * a.p.three_body_weight, hd3 = -0.5f * a.p.three_body_decay;
    const float4* rA = reinterpret_cast<const float4*>(recA);
    const float4* rB = reinterpret_cast<const float4*>(recB);
    const float4* tab = reinterpret_cast<const float4*>(trip);
    const int ntrip = nn * (nn - 1) / 2;

    const bool whole = ntrip <= a.tcap;
    for (int t0 = 0; t0 < ntrip; t0 += a.tcap) {
        const int t1 = min(t0 + a.tcap, ntrip);
        if (t0 > 0) __syncthreads();                     // the previous chunk has been read
        for (int tt = t0 + tid; tt < t1; tt += NT) {
            int j, k;
            if (whole) unrank_pair_kmajor(tt, j, k);     // any order of filling does
            else unrank_triple(goff, pbase, ns, np, tt, j, k);
            const float4 Aj = rA[j], Ak = rA[k], Bj = rB[j], Bk = rB[k];
            const int to = whole ? triple_place(pbase, ns, Bj, Bk) : tt - t0;
            float4 entry = table_entry(zw3, hd3, Aj, Bj, Ak, Bk);
            if constexpr (LEAN) entry.w = group_ratio<18>(h, entry.x);
            reinterpret_cast<float4*>(trip)[to] = entry;
        }
        __syncthreads();
        // this wavefront's share of the chunk: a run of consecutive entries, which meets few element pairs
        const int len = t1 - t0, w0 = len * wave / NW, w1 = len * (wave + 1) / NW;
        int pq = 0;
        while (pq < np - 1 && pbase[pq + 1] - t0 <= w0) ++pq;
        for (; pq < np && pbase[pq] - t0 < w1; ++pq) {
            const int s0 = __builtin_amdgcn_readfirstlane(max(pbase[pq] - t0, w0));
            const int count = __builtin_amdgcn_readfirstlane(min(pbase[pq + 1] - t0, w1)) - s0;
            if (count <= 0) continue;
            const int rounds = idiv_small(count, TS), rest = count - rounds * TS;
            const float4* src = tab + s0 + (tsub < TS ? tsub : 0);
            float* dst = part + ((size_t)pq * NW + wave) * per;
            if constexpr (LEAN) {
                float v[4] = {0.f, 0.f, 0.f, 0.f};
                auto add = [&](const float4* at, auto even) {
                    const float4 t = *at;
                    const float d0 = t.x - rsl[0], d1 = t.x - rsl[1];
                    const float e0 = fexp2(-d0 * d0), e1 = decltype(even)::value ? e0 * t.w : fexp2(-d1 * d1);
                    v[0] = fmaf(e0, t.y, v[0]);
                    v[1] = fmaf(e0, t.z, v[1]);
                    v[2] = fmaf(e1, t.y, v[2]);
                    v[3] = fmaf(e1, t.z, v[3]);
                };
                auto run = [&](auto even) {
#pragma unroll 2
                    for (int it = 0; it < rounds; ++it) add(src + it * LEAN_SLOTS, even);
                    if (rest > 0) add(tsub < rest ? src + rounds * LEAN_SLOTS : tab + a.tcap, even);
                };
                if (h != 0.0f) run(std::true_type{});
                else run(std::false_type{});
                v[2] *= factor;
                v[3] *= factor;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    v[c] += __shfl(v[c], lane + 30, 64);
                    v[c] += __shfl(v[c], lane + 10, 64) + __shfl(v[c], lane + 20, 64);
                }
                if (tsub == 0) {                         // this wavefront's words alone
                    if (2 * ll < nRs3) dst[4 * ll] += v[0], dst[4 * ll + 1] += v[1];
                    if (2 * ll + 1 < nRs3) dst[4 * ll + 2] += v[2], dst[4 * ll + 3] += v[3];
                }
                continue;
            }
#pragma unroll
            for (int b = 0; b < MAXLB; ++b) {
                if (b * 64 < nRs3) {
                    float c_ = 0.0f, s_ = 0.0f;
#pragma unroll 4
                    for (int it = 0; it < rounds; ++it) {
                        const float3v v = *reinterpret_cast<const float3v*>(src + it * TS);
                        const float d = v.x - rsl[b];
                        const float e = fexp2(-d * d);
                        c_ = fmaf(e, v.y, c_);
                        s_ = fmaf(e, v.z, s_);
                    }
                    if (rest > 0) {
                        const float3v v = *reinterpret_cast<const float3v*>(tsub < rest ? src + rounds * TS : tab + a.tcap);
                        const float d = v.x - rsl[b];
                        const float e = fexp2(-d * d);
                        c_ = fmaf(e, v.y, c_);
                        s_ = fmaf(e, v.z, s_);
                    }
                    float tc = c_, tsn = s_;
                    for (int k = 1; k < TS; ++k) {
                        tc += __shfl(c_, ll + W3 * k, 64);
                        tsn += __shfl(s_, ll + W3 * k, 64);
                    }
                    const int l = b * 64 + ll;
                    if (tsub == 0 && l < nRs3) {          // this wavefront's words alone
                        dst[2 * l] += tc;
                        dst[2 * l + 1] += tsn;
                    }
                }
            }
        }
    }
    if constexpr (NW == 1) return;
    __syncthreads();
    // the partial blocks, wavefront by wavefront; the pairs' blocks of the row follow each other in this order
    float* out3 = out + ns * nRs2;
    for (int t = tid; t < np * per; t += NT) {
        const int pq = idiv_small(t, per), x = t - pq * per;
        const float* src = part + (size_t)pq * NW * per + x;
        float v = src[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += src[w * per];
        out3[t] = v;
    }
}

// ---------------------------------------------------------------------------------
// d/dr of the two-body bin values of one neighbour, contracted or not
// ---------------------------------------------------------------------------------
struct TwoBody {
    float mu, s2, s2p, mup, pre, fc, dfc, d2_over_r;
};

__device__ __forceinline__ TwoBody two_body_setup(float r, float fc, float dfc, const qmll_fchl_params& p) {
    TwoBody t;
    const float r2 = r * r;
    t.s2 = flog(1.0f + p.eta2 * frcp(r2));
    t.mu = flog(r) - 0.5f * t.s2;
    t.s2p = -2.0f * p.eta2 * frcp(r * (r2 + p.eta2));      // d sigma^2 / dr
    t.mup = frcp(r) - 0.5f * t.s2p;                   // d mu / dr
    t.pre = frsq(t.s2) * 0.3989422804014327f * fexp2(-p.two_body_decay * flog2(r));
    t.fc = fc;
    t.dfc = dfc;
    t.d2_over_r = p.two_body_decay * frcp(r);
    return t;
}

// value and r-derivative of bin z
__device__ __forceinline__ void two_body_bin(const TwoBody& t, float lnRs, float invRs, float& val, float& dval) {
    const float u = lnRs - t.mu;
    const float inv_s2 = frcp(t.s2);
    const float Bz = t.pre * invRs * fexp2(-0.5f * LOG2E * u * u * inv_s2);
    const float Q = -0.5f * t.s2p * inv_s2 - t.d2_over_r + u * inv_s2 * (t.mup + 0.5f * u * t.s2p * inv_s2);
    val = Bz * t.fc;
    dval = Bz * (t.fc * Q + t.dfc);
}

// partial derivatives with respect to (a,b,c) of the triple's prefactor
// K = w3 (1 + 3 ci cj ck) (abc)^-d3 fc(a) fc(b), and of cos_i
struct TripleDeriv {
    float K, Ka, Kb, Kc;     // K and its partials
    float cia, cib, cic;     // partials of cos_i
};

__device__ __forceinline__ TripleDeriv triple_derivatives(const Triple& t, const qmll_fchl_params& p, float fa,
                                                          float dfa, float fb, float dfb) {
    TripleDeriv d;
    const float ia = frcp(t.a), ib = frcp(t.b), ic = frcp(t.c);
    // d cos / d distance (law of cosines)
    d.cia = ib - t.ci * ia;
    d.cib = ia - t.ci * ib;
    d.cic = -t.c * ia * ib;
    const float cja = ic - t.cj * ia, cjb = -t.b * ia * ic, cjc = ia - t.cj * ic;
    const float cka = -t.a * ib * ic, ckb = ic - t.ck * ib, ckc = ib - t.ck * ic;
    const float P = 1.0f + 3.0f * t.ci * t.cj * t.ck;
    const float Pa = 3.0f * (d.cia * t.cj * t.ck + t.ci * cja * t.ck + t.ci * t.cj * cka);
    const float Pb = 3.0f * (d.cib * t.cj * t.ck + t.ci * cjb * t.ck + t.ci * t.cj * ckb);
    const float Pc = 3.0f * (d.cic * t.cj * t.ck + t.ci * cjc * t.ck + t.ci * t.cj * ckc);
    const float dec = p.three_body_weight * fexp2(-p.three_body_decay * flog2(t.a * t.b * t.c));
    const float ksi = dec * P;
    const float ksia = dec * (Pa - p.three_body_decay * P * ia);
    const float ksib = dec * (Pb - p.three_body_decay * P * ib);
    const float ksic = dec * (Pc - p.three_body_decay * P * ic);
    d.K = ksi * fa * fb;
    d.Ka = ksia * fa * fb + ksi * dfa * fb;
    d.Kb = ksib * fa * fb + ksi * fa * dfb;
    d.Kc = ksic * fa * fb;
    return d;
}

// copies of the neighbours' force array that one wavefront of the backward kernel needs for nn neighbours: as many
// s = tt / nn as 64 consecutive triple numbers tt span, and at least one for the two-body part
__host__ __device__ __forceinline__ int force_copies(int nn) {
    if (nn < 2) return 1;
    const int span = (62 + nn) / nn + 1, all = nn / 2;
    return span < all ? span : all;
}

// ---------------------------------------------------------------------------------
// VJP
// ---------------------------------------------------------------------------------
// The forces of a triple on its two neighbours are added into LDS without atomics (ds_add_f32 costs tens of clocks
// PER LANE here: with them 16 boxes of 96 atoms took 190 us, with their adds taken out 54): the triples are numbered so
// that consecutive lanes have different j and different k, and a wavefront keeps as many private copies of the
// neighbours' force array as 64 consecutive triples can meet the same neighbour (force_copies).  An instruction's lanes then
// read, add and write different words, one 16-byte record each, and the copies are summed at the end.  NW wavefronts
// per atom share out the triples: see wavefronts_backward.
// COMPACT (one wavefront): the form for capacities at which the copies above do not fit.  [cap] records of three floats hold
// as many copies as the atom's own neighbours leave room for, at least one; where an instruction's lanes would need more, its
// s-rows take turns.
// LEAN: grids of LEAN_RS3 - 3 .. LEAN_RS3 bins, on scalar registers, as in fchl19_vjp_lean_kernel
template <int NW, bool COMPACT = false, bool LEAN = false>
__global__ __launch_bounds__(64 * NW) void fchl19_vjp_kernel(FchlArgs a, const float* __restrict__ grad_rep,
                                                              float* __restrict__ grad_X) {
    extern __shared__ float smem[];
    constexpr int NT = 64 * NW;
    const int tid = threadIdx.x, lane = NW == 1 ? tid : tid & 63;
    const int wave = NW == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = a.molIDs[blockIdx.x];
    const int i = a.atomIDs[blockIdx.x];
    if (m < 0 || m >= a.B || i < 0 || i >= a.n) return;   // malformed index: write nothing
    const int ns = a.p.nspecies, nRs2 = a.p.nRs2, nRs3 = a.p.nRs3;
    const int R2 = ns * nRs2;                        // two-body part of a representation row
    const int row3 = LEAN ? LEAN_RS3 : nRs3;         // an element pair's entries as they are staged
    const int NE3 = (ns * (ns + 1) / 2) * row3;      // (element pair, radial bin) entries of its three-body part

    // [cap][4] per neighbour, read with one instruction each: (d_ij, r) and
    // (1 / r, fc, dfc / dr, element type); first in LDS, 16-byte aligned
    float* recA = smem;
    float* recB = recA + 4 * a.cap;
    static_assert(!COMPACT || NW == 1, "the compact force records belong to one wavefront");
    constexpr int FR = COMPACT ? 3 : 4;        // floats per force record
    // [NW][tcap][FR] forces on the neighbours: copies of nn records (compact: behind gin3, which the 16-byte records precede)
    float* force = recB + 4 * a.cap + (COMPACT ? 2 * NE3 : 0);
    float* gin3 = COMPACT ? recB + 4 * a.cap : force + FR * NW * a.tcap;   // [NE3][2] incoming gradient of the three-body bins
                                                                           // (cos, sin), see below; 8-byte aligned
    int* sj = (int*)(COMPACT ? force + FR * a.tcap : gin3 + 2 * NE3);      // [cap] atom index of neighbour j
    int* goff = sj + a.cap;              // [ns+1] slices of the sorted neighbour list by type
    int* wcount = goff + ns + 1;         // [ns * NW] scratch of the staging
    float* slnRs2 = (float*)(wcount + (NW > 1 ? ns * NW : 0));   // [nRs2]
    float* sRs3 = slnRs2 + nRs2;     // [nRs3] sk3 Rs3 (fast form: about the middle of the grid)
    float* sfac = sRs3 + nRs3;       // [nRs3] 2^(-u^2) of every bin (fast form)
    float* gin2 = sfac + nRs3;       // [R2] incoming gradient of the two-body bins, each divided by its Rs2
    const float4* rA = reinterpret_cast<const float4*>(recA);
    const float4* rB = reinterpret_cast<const float4*>(recB);

    // Global loads that do not depend on the neighbourhood (grid tables, the incoming gradient
    // row) are issued first and consumed after the staging, so their latency overlaps the
    // staging's own loads.
    const float* gsrc = grad_rep + ((size_t)m * a.n + i) * (R2 + ns * (ns + 1) * nRs3);
    // entry e of the three-body part in the incoming row; negative: a bin that is not there
    auto source3 = [&](int e) {
        if (!LEAN) return e;
        const int pq = idiv_small(e, LEAN_RS3), l = e - pq * LEAN_RS3;
        return l < nRs3 ? __mul24(pq, nRs3) + l : -1;
    };
    constexpr int GREG2 = NW > 2 ? 1 : 2, GREG3 = NW > 2 ? 1 : 4 / NW;   // values / (cos, sin) pairs per thread held in registers
    float gr2[GREG2], gr3c[GREG3], gr3s[GREG3];
#pragma unroll
    for (int k = 0; k < GREG2; ++k) gr2[k] = tid + NT * k < R2 ? gsrc[tid + NT * k] : 0.0f;
#pragma unroll
    for (int k = 0; k < GREG3; ++k) {
        const int e = tid + NT * k;
        const int from = e < NE3 ? source3(e) : -1;
        gr3c[k] = from >= 0 ? gsrc[R2 + 2 * from] : 0.0f;
        gr3s[k] = from >= 0 ? gsrc[R2 + 2 * from + 1] : 0.0f;
    }
    const float rs2v = lane < nRs2 ? a.Rs2[lane] : 1.0f;
    const float rs3v = lane < nRs3 ? a.Rs3[lane] : 0.0f;
    float* mine = force + FR * wave * a.tcap;   // this wavefront's copies
    auto set_force = [&](float* p, float x, float y, float z) {
        if constexpr (COMPACT) p[0] = x, p[1] = y, p[2] = z;
        else *reinterpret_cast<float4*>(p) = make_float4(x, y, z, 0.0f);
    };
    auto add_force = [&](float* p, float x, float y, float z) {
        float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
        if constexpr (COMPACT) f.x = p[0], f.y = p[1], f.z = p[2];
        else f = *reinterpret_cast<float4*>(p);
        f.x += x;
        f.y += y;
        f.z += z;
        if constexpr (COMPACT) set_force(p, f.x, f.y, f.z);
        else *reinterpret_cast<float4*>(p) = f;
    };
    for (int t = lane; t < a.tcap; t += QMLL_WAVE) set_force(mine + FR * t, 0.f, 0.f, 0.f);
    const float inv_rc = frcp(a.p.rcut);
    auto emit = [&](int pos, int, int, int e, int j, float dx, float dy, float dz, float r2) {
        const float ir = __builtin_amdgcn_rsqf(r2), r = root(r2, ir);
        float fc, dfc;
        cutoff(r, inv_rc, fc, dfc);
        reinterpret_cast<float4*>(recA)[pos] = make_float4(dx, dy, dz, r);
        reinterpret_cast<float4*>(recB)[pos] = make_float4(ir, fc, dfc, __int_as_float(e));
        sj[pos] = j;
    };
    int nn;
    if constexpr (NW == 1) nn = visit_neighbours(a, goff, m, i, lane, emit);
    else nn = visit_neighbours_wide<NW>(a, goff, wcount, m, i, tid, emit);
    const float k3 = a.p.eta3 * LOG2E;
    const float sk3 = fsqrt(k3);                       // the radial grid of the triples is kept as sk3 Rs3
    const float hfac = -2.0f * a.p.eta3 * frcp(sk3);
    // The radial factor of a triple, exp2(-(x - g_l)^2) with x = sk3 rho and g_l = sk3 Rs3_l, about the
    // middle of the grid (y = x - mid, u_l = g_l - mid): exp2(2 y u_l - y^2) 2^(-u_l^2).  The second
    // factor does not depend on the triple and goes into the staged gradient once per atom; the first
    // is one fma and the exponential per (triple, bin).  It is at most 2^(u_l^2), so the form is taken
    // only while u_l^2 <= 100 for every bin (eta3 rcut^2 up to about 270); beyond, the plain form runs.
    // LEAN: see group_sums; where the grid is not even, the plain form.
    const float mid = 0.5f * sk3 * a.p.rcut;
    const float ul = LEAN && lane < nRs3 ? fmaf(sk3, rs3v, -mid) : 0.0f;
    bool stops = false;
    const float spacing = LEAN ? even_spacing(ul, lane, lane < nRs3, nRs3, mid, a.nlist ? LINE_ANY : LINE_WITHIN, stops) : 0.0f;
    const bool even = LEAN && spacing != 0.0f;
    bool fast = false;
    if constexpr (!LEAN) {
        float um = fabsf(fmaf(sk3, rs3v, -mid));
        if (lane >= nRs3) um = 0.0f;
        for (int t = lane + QMLL_WAVE; t < nRs3; t += QMLL_WAVE) um = fmaxf(um, fabsf(fmaf(sk3, a.Rs3[t], -mid)));
        um = fmaxf(um, lane_xor<1>(um));
        um = fmaxf(um, lane_xor<2>(um));
        um = fmaxf(um, lane_xor<4>(um));
        um = fmaxf(um, lane_xor<8>(um));
        um = fmaxf(um, lane_xor<16>(um));
        um = fmaxf(um, lane_xor<32>(um));
        fast = __builtin_amdgcn_readfirstlane(__float_as_int(um)) <= __float_as_int(10.0f);
    }
    const float shift = LEAN || fast ? mid : 0.0f;
    // the gradient of the two-body bins, each divided by its grid point (the bin's 1 / Rs2 factor)
#pragma unroll
    for (int k = 0; k < GREG2; ++k) {
        const int t = tid + NT * k;
        if (t < R2) gin2[t] = gr2[k] * (a.gscale * frcp(a.Rs2[t - nRs2 * idiv_small(t, nRs2)]));
    }
    for (int t = tid + NT * GREG2; t < R2; t += NT)
        gin2[t] = gsrc[t] * (a.gscale * frcp(a.Rs2[t - nRs2 * idiv_small(t, nRs2)]));
    if (lane < nRs2 && wave == 0) slnRs2[lane] = flog(rs2v);
    for (int t = tid + QMLL_WAVE; t < nRs2; t += NT) slnRs2[t] = flog(a.Rs2[t]);
    if constexpr (LEAN) {
        const float f = a.gscale * (even ? group_factor(ul, lane, lane, spacing) : 1.0f);
        if (tid < nRs3) sfac[tid] = f;
    }
    for (int t = LEAN ? nRs3 : tid; t < nRs3; t += NT) {
        const float u = fmaf(sk3, t == lane ? rs3v : a.Rs3[t], -shift);
        sRs3[t] = u;
        sfac[t] = a.gscale * (fast ? fexp2(-u * u) : 1.0f);
    }
    __syncthreads();
    // the gradient of the three-body bins per (element pair, radial bin), (cos, sin) parts, times the
    // bin's constant factor s = 2^(-u^2): with e' = exp2(2 y u - y^2) the sums over the bins of g e and
    // of g (x - g_l) e are sum (g s) e' and y sum (g s) e' - sum (g s) (u e')
    auto stage3 = [&](int e, float gc, float gs) {
        const int l = e - row3 * idiv_small(e, row3);
        const float s_ = sfac[LEAN ? min(l, nRs3 - 1) : l];
        reinterpret_cast<float2*>(gin3)[e] = make_float2(gc * s_, gs * s_);
    };
#pragma unroll
    for (int k = 0; k < GREG3; ++k)
        if (tid + NT * k < NE3) stage3(tid + NT * k, gr3c[k], gr3s[k]);
    for (int e = tid + NT * GREG3; e < NE3; e += NT) {
        const int from = source3(e);
        stage3(e, from >= 0 ? gsrc[R2 + 2 * from] : 0.0f, from >= 0 ? gsrc[R2 + 2 * from + 1] : 0.0f);
    }
    __syncthreads();

    float gix = 0.0f, giy = 0.0f, giz = 0.0f;

    // two-body: lanes = (bin group g, neighbour j); group g takes the bins z = g, g+G, ...
    // With u = ln Rs - mu the r-derivative of a bin is B_z (fc Q + dfc), B_z = pre / Rs exp2(-c u^2) and
    // Q a quadratic in u whose coefficients (and fc, dfc) depend on the neighbour only:
    // per bin a subtraction, the exponential and two fma for the quadratic.
    {
        const int G = (nn > 0 && nn < 64) ? idiv_small(64, nn) : 1;
        for (int base = 0; base < nn; base += QMLL_WAVE) {
            const int g = G > 1 ? idiv_small(lane, nn) : 0;
            const int j = G > 1 ? lane - g * nn : base + lane;
            const bool active = g < G && j < nn;
            float gr = 0.0f;
            float4 Aj = make_float4(0.f, 0.f, 0.f, 1.f), Bj = make_float4(1.f, 0.f, 0.f, 0.f);
            if (active) {
                Aj = rA[j];
                Bj = rB[j];
                const TwoBody tb = two_body_setup(Aj.w, Bj.y, Bj.z, a.p);
                const float inv_s2 = frcp(tb.s2);
                const float nc = -0.5f * LOG2E * inv_s2;
                const float hs = 0.5f * tb.s2p * inv_s2;
                const float q0 = fmaf(tb.fc, -hs - tb.d2_over_r, tb.dfc);
                const float q1 = tb.fc * inv_s2 * tb.mup;
                const float q2 = tb.fc * hs * inv_s2;
                const float* gz = gin2 + __float_as_int(Bj.w) * nRs2;
                for (int z = g + G * wave; z < nRs2; z += G * NW) {
                    const float u = slnRs2[z] - tb.mu;
                    const float e = fexp2(u * u * nc);
                    gr = fmaf(gz[z] * e, fmaf(fmaf(q2, u, q1), u, q0), gr);
                }
                gr *= tb.pre;
            }
            float tot = gr;
            for (int k = 1; k < G; ++k) tot += __shfl(gr, (lane + nn * k) & 63, 64);
            if (active && g == 0) {
                const float ux = Aj.x * Bj.x, uy = Aj.y * Bj.x, uz = Aj.z * Bj.x;   // dr/dR_i
                gix += tot * ux;
                giy += tot * uy;
                giz += tot * uz;
                set_force(mine + FR * j, -tot * ux, -tot * uy, -tot * uz);   // each lane owns its own j here
            }
        }
    }
    __syncthreads();

    // three-body: lane per triple, serial over radial bins.  With a = d_ij, b = d_ik, c = b - a
    // (= R_j - R_k) and X = cos_i cos_j cos_k the partials of P = 1 + 3 X by the three distances
    // follow from the law of cosines:
    //   P_a / 3 = cos_j cos_k / |b| + cos_i cos_k / |c| - cos_i cos_j |a| / (|b| |c|) - 2 X / |a|
    // and cyclically; K = w3 P (abc)^-d3 fc(a) fc(b) and its partials share the factor
    // dec = w3 (abc)^-d3, applied once at the end together with 2 exp(-pi^2 / 2).
    const int ntrip = nn * (nn - 1) / 2;
    const float zeta2 = 0.014383766711652736f;   // 2 exp(-pi^2 / 2)
    const float d3 = a.p.three_body_decay;
    float us[LEAN ? LEAN_RS3 : 1], ratio[LEAN_RS3 / RS3_GROUP];        // the grid, on scalar registers
    if constexpr (LEAN) {
        const float v = group_ratio<0>(-spacing, ul);
#pragma unroll
        for (int l = 0; l < LEAN_RS3; ++l) us[l] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ul), l));
#pragma unroll
        for (int q = 0; q < LEAN_RS3 / RS3_GROUP; ++q) ratio[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), RS3_GROUP * q));
    }
    // copies of the force records that this atom uses: one for every s-row of an instruction, or as many as there is room for
    auto copies = [&] { return COMPACT ? min(force_copies(nn), idiv_small(a.tcap, max(nn, 1))) : force_copies(nn); };
    for (int tt = tid; tt < ntrip; tt += NT) {
        // tt = s nn + j: the pair {j, j + s + 1 mod nn} (when nn is even, the first half of the last s)
        const int s = idiv_small(tt, nn), j = tt - __mul24(s, nn);
        int k = j + s + 1;
        if (k >= nn) k -= nn;
        // the copy: 64 consecutive tt meet a neighbour once per s
        const int row = s - idiv_small(tt - lane, nn);
        const int turn = COMPACT ? idiv_small(row, copies()) : 0;
        float* own = mine + FR * __mul24(COMPACT ? row - __mul24(turn, copies()) : row, nn);
        const float4 Aj = rA[j], Ak = rA[k], Bj = rB[j], Bk = rB[k];
        const float ia = Bj.x, ib = Bk.x;
        const float cx = Ak.x - Aj.x, cy = Ak.y - Aj.y, cz = Ak.z - Aj.z;
        const float c2 = cx * cx + cy * cy + cz * cz;
        const float ic = __builtin_amdgcn_rsqf(c2), c = c2 * ic;
        const float vi = Aj.x * Ak.x + Aj.y * Ak.y + Aj.z * Ak.z;
        const float dac = Aj.x * cx + Aj.y * cy + Aj.z * cz;
        const float dcb = cx * Ak.x + cy * Ak.y + cz * Ak.z;
        const float w = ia * ib, iaic = ia * ic, ibic = ib * ic;
        const float ci = vi * w, cj = -dac * iaic, ck = dcb * ibic;
        // a^2 b^2 - (d_ij.d_ik)^2 = |d_ij x d_ik|^2 (Lagrange): the cross product keeps full
        // relative accuracy near collinear triples, where the difference of squares cancels
        const float px = Aj.y * Ak.z - Aj.z * Ak.y, py = Aj.z * Ak.x - Aj.x * Ak.z, pz = Aj.x * Ak.y - Aj.y * Ak.x;
        const float cross2 = px * px + py * py + pz * pz;
        const float cosT = fminf(1.0f, fmaxf(-1.0f, ci));
        const float sinT = fminf(1.0f, fsqrt(cross2) * w);
        const float guard_inv = Aj.w * Ak.w * __builtin_amdgcn_rsqf(fmaxf(1e-10f, cross2));
        const float q1 = cj * ck, q2 = ci * ck, q3 = ci * cj;
        const float X = ci * q1, X2 = X + X;
        const float P = fmaf(3.0f, X, 1.0f);
        const float Pa3 = fmaf(q1, ib, fmaf(q2, ic, fmaf(-q3 * Aj.w, ibic, -X2 * ia)));
        const float Pb3 = fmaf(q1, ia, fmaf(q3, ic, fmaf(-q2 * Ak.w, iaic, -X2 * ib)));
        const float Pc3 = fmaf(q2, ia, fmaf(q3, ib, fmaf(-q1 * c, w, -X2 * ic)));
        const float Z = zeta2 * a.p.three_body_weight * fexp2(-d3 * flog2(Aj.w * Ak.w * c));
        const float fa = Bj.y, dfa = Bj.z, fb = Bk.y, dfb = Bk.z;
        const float F = fa * fb, d3P = d3 * P, FP = F * P;
        const float ka = fmaf(F, fmaf(3.0f, Pa3, -d3P * ia), P * dfa * fb);   // K_a / dec
        const float kb = fmaf(F, fmaf(3.0f, Pb3, -d3P * ib), P * fa * dfb);
        const float kc = F * fmaf(3.0f, Pc3, -d3P * ic);
        // the (element pair, radial bin) entries of this triple's pair
        const int tj = __float_as_int(Bj.w), tk = __float_as_int(Bk.w);
        const int tp = min(tj, tk), tq = max(tj, tk);
        const float2* g = reinterpret_cast<const float2*>(gin3) + __mul24(row3, __mul24(ns, tp) - (__mul24(tp, tp + 1) >> 1) + tq);
        // exp(-eta3 (rho - Rs)^2) = exp2(-(x - g_l)^2), x = sk3 rho, the grid stored pre-scaled;
        // d e / d rho = -2 eta3 (rho - Rs) e = hfac (x - g_l) e, the factor applied after the sums
        const float y = fmaf(sk3 * 0.5f, Aj.w + Ak.w, -shift);
        float Gc = 0.f, Gs = 0.f, Hc = 0.f, Hs = 0.f;
        auto bins = [&](auto bin) {
            if constexpr (LEAN) {
#pragma unroll
                for (int l = 0; l < LEAN_RS3; l += 2) {
                    const float4 gv = reinterpret_cast<const float4*>(g)[l / 2];
                    bin(gv.x, gv.y, us[l]);
                    bin(gv.z, gv.w, us[l + 1]);
                }
            } else {
#pragma unroll 4
                for (int l = 0; l < nRs3; ++l) bin(g[l].x, g[l].y, sRs3[l]);
            }
        };
        auto groups = [&](float B, auto stop) {
#pragma unroll
            for (int q = 0; q < LEAN_RS3 / RS3_GROUP; ++q) {
                const float d = y - us[LEAN ? RS3_GROUP * q : 0], Q = B * ratio[q];
                group_sums(g + RS3_GROUP * q, d, fexp2(-(d * d)), decltype(stop)::value ? fminf(Q, RATIO_STOP) : Q, spacing, Gc, Gs, Hc, Hs);
            }
        };
        if (__builtin_expect(even && !stops, 1)) {
            groups(group_ratio<18>(spacing, y), std::false_type{});
        } else if (even) {
            groups(group_ratio<100>(spacing, y), std::true_type{});
        } else if (fast) {
            const float y2 = y + y, ny2 = -y * y;
            bins([&](float gc, float gs, float u) {
                const float e = fexp2(fmaf(y2, u, ny2));
                const float ue = u * e;
                Gc = fmaf(gc, e, Gc);
                Gs = fmaf(gs, e, Gs);
                Hc = fmaf(gc, ue, Hc);
                Hs = fmaf(gs, ue, Hs);
            });
            Hc = fmaf(y, Gc, -Hc);
            Hs = fmaf(y, Gs, -Hs);
        } else {
            bins([&](float gc, float gs, float u) {
                const float dl = y - u;
                const float e = fexp2(-(dl * dl));
                const float de = dl * e;
                Gc = fmaf(gc, e, Gc);
                Gs = fmaf(gs, e, Gs);
                Hc = fmaf(gc, de, Hc);
                Hs = fmaf(gs, de, Hs);
            });
        }
        const float S0 = Gc * cosT + Gs * sinT;
        const float S1 = 0.5f * hfac * (Hc * cosT + Hs * sinT);                   // d rho/da = d rho/db = 1/2
        const float Sth = (Gc * sinT - Gs * cosT) * guard_inv;                     // multiplies d cos_i
        // d cos_i / d distance: 1/b - cos_i / a, 1/a - cos_i / b, -c / (a b)
        const float ea = Z * ia * fmaf(ka, S0, FP * fmaf(Sth, fmaf(-ci, ia, ib), S1));   // (d L / d a) / a
        const float eb = Z * ib * fmaf(kb, S0, FP * fmaf(Sth, fmaf(-ci, ib, ia), S1));
        const float ec = Z * ic * fmaf(kc, S0, -FP * Sth * c * w);
        gix = fmaf(ea, Aj.x, fmaf(eb, Ak.x, gix));
        giy = fmaf(ea, Aj.y, fmaf(eb, Ak.y, giy));
        giz = fmaf(ea, Aj.z, fmaf(eb, Ak.z, giz));
        // force on j: ec (d_ik - d_ij) - ea d_ij, on k: -ec (d_ik - d_ij) - eb d_ik
        const float jx = fmaf(ec, cx, -ea * Aj.x), jy = fmaf(ec, cy, -ea * Aj.y), jz = fmaf(ec, cz, -ea * Aj.z);
        const float kx = fmaf(-ec, cx, -eb * Ak.x), ky = fmaf(-ec, cy, -eb * Ak.y), kz = fmaf(-ec, cz, -eb * Ak.z);
        const int turns = COMPACT ? idiv_small(force_copies(nn) + copies() - 1, copies()) : 1;
        for (int now = 0; now < turns; ++now) {
            if (!COMPACT || now == turn) {
                add_force(own + FR * j, jx, jy, jz);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the next read sees every lane's write (LDS instructions run in order)
                add_force(own + FR * k, kx, ky, kz);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    __syncthreads();
    gix = wave_sum(gix);
    giy = wave_sum(giy);
    giz = wave_sum(giz);
    float* gm = grad_X + (size_t)m * a.n * 3;
    if (lane == 0) {
        atomicAdd(&gm[i * 3 + 0], gix);
        atomicAdd(&gm[i * 3 + 1], giy);
        atomicAdd(&gm[i * 3 + 2], giz);
    }
    const int ncopies = copies();
    for (int it = tid; it < 3 * nn; it += NT) {
        const int x = idiv_small(it, 3), c = it - 3 * x;
        float sum = 0.0f;
        for (int w = 0; w < NW; ++w)
            for (int q = 0; q < ncopies; ++q) sum += force[FR * (w * a.tcap + q * nn + x) + c];
        atomicAdd(&gm[sj[x] * 3 + c], sum);
    }
}

// ---------------------------------------------------------------------------------
// VJP, one wavefront per central atom, number of elements known to the compiler
//
// The same sums as fchl19_vjp_kernel<1> where fchl19_forward_lean_kernel has those of the forward kernel, and for the same reasons:
// that kernel takes 1640 vector, 434 scalar and 137 LDS instructions per atom of 20 neighbours, and its bin loop reads 12 bytes per lane and
// bin, six clocks of the LDS that four SIMDs share.  Here the grid is on scalar registers, the two bins of a 16-byte read are unrolled
// with their places as constants, a lane stages the gradient of one radial bin of three pairs at a time (its constant factor is then in
// a register), and the number of a triple's pair comes from the neighbours' records in two instructions: 1426 + 288 + 98 instructions
// (before the bins were taken in groups).  86016 atoms of 21, three elements 193 -> 165 us, 131235 atoms of 3 to 29, five elements
// 342 -> 290, 64000 of 8 89 -> 63, 80000 of 40 476 -> 446.  Vector issue takes five sixths of the launch.
// ---------------------------------------------------------------------------------
// NW > 1: the wavefronts of the workgroup share the triples (and have copies of the forces each); gradient() is then called, by all of them,
// when the neighbours are staged, and returns the atom's row of the incoming gradient.
template <int NS, int NW, class Gradient>
__device__ __forceinline__ void lean_vjp(const FchlArgs& a, int m, int i, float* smem, Gradient&& gradient, float* __restrict__ grad_X) {
    constexpr int NP = NS * (NS + 1) / 2;
    constexpr int STEP = 3 * LEAN_RS3;                   // entries of the gradient's three-body part per load of the wavefront
    constexpr bool ONE = NW == 1;
    const int lane = ONE ? threadIdx.x : threadIdx.x & 63, wave = ONE ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nRs2 = a.p.nRs2, nRs3 = a.p.nRs3;
    float* recA = smem;                                  // [cap][4]: d_ij, r
    float* recB = recA + 4 * a.cap;                      // [cap][4]: 1 / r, fc, dfc / dr, the type's pairs (below)
    float* force = recB + 4 * a.cap;                     // [NW][tcap][4] forces on the neighbours, in copies
    float* gin3 = force + 4 * NW * a.tcap;               // [NP][LEAN_RS3][2] incoming gradient of the three-body bins
    float* gin2 = gin3 + 2 * NP * LEAN_RS3;              // [NS][32] and of the two-body ones, each divided by its Rs2
    float* slnRs2 = gin2 + 32 * NS;                      // [32]
    int* sj = (int*)(slnRs2 + 32);                       // [cap] atom index of neighbour j
    float* own_force = reinterpret_cast<float*>(sj + a.cap);       // NW > 1: [NW][3], what the wavefronts have for atom i itself
    float* mine = force + 4 * wave * a.tcap;

    const float* Xm = a.X + (size_t)m * a.n * 3;
    const int own = lane < a.n ? lane : 0;
    const float xo = Xm[own * 3 + 0], yo = Xm[own * 3 + 1], zo = Xm[own * 3 + 2];
    const int et = a.types[(size_t)m * a.n + own];
    const int total = min(a.natoms[m], a.n);
    const int z = lane & 31;
    const float rs2v = z < nRs2 ? a.Rs2[z] : 1.0f;
    // three pairs' bins at a time: a lane has the same bin each time
    const int third = idiv_small(lane, LEAN_RS3), l3 = lane - LEAN_RS3 * third;
    const bool bin_ok = lane < STEP && l3 < nRs3;
    const float rs3v = bin_ok ? a.Rs3[l3] : 0.0f;
    const float* gsrc = nullptr;
    if constexpr (ONE) gsrc = gradient();
    float g2[(NS + 1) / 2];
#pragma unroll
    for (int k = 0; k < (NS + 1) / 2; ++k) {
        const int e = 2 * k + (lane >> 5);
        g2[k] = ONE && e < NS && z < nRs2 ? gsrc[e * nRs2 + z] : 0.0f;
    }
    float2 g3[(NP + 2) / 3];
#pragma unroll
    for (int k = 0; k < (NP + 2) / 3; ++k) {
        g3[k] = make_float2(0.f, 0.f);
        if (ONE && bin_ok && 3 * k + third < NP) __builtin_memcpy(&g3[k], gsrc + NS * nRs2 + 2 * ((3 * k + third) * nRs3 + l3), 8);
    }
    for (int t = lane; t < a.tcap; t += QMLL_WAVE) reinterpret_cast<float4*>(mine)[t] = make_float4(0.f, 0.f, 0.f, 0.f);

    const float inv_rc = frcp(a.p.rcut);
    const float sk3 = fsqrt(a.p.eta3 * LOG2E);
    const float hfac = -2.0f * a.p.eta3 * frcp(sk3);
    const float mid = 0.5f * sk3 * a.p.rcut;             // distances and bins about the middle of the range: half the rounding
    const float ul = bin_ok ? fmaf(sk3, rs3v, -mid) : 0.0f;
    bool stops;
    const float spacing = even_spacing(ul, l3, bin_ok, nRs3, mid, LINE_WITHIN, stops);
    const bool even = spacing != 0.0f;

    // ---- neighbours: candidate = lane ----
    float dx = Xm[i * 3 + 0] - xo, dy = Xm[i * 3 + 1] - yo, dz = Xm[i * 3 + 2] - zo;
    if (a.cell != nullptr) min_image(dx, dy, dz, a.cell + (size_t)m * 9, a.inv_cell + (size_t)m * 9);
    const float r2 = dx * dx + dy * dy + dz * dz;
    const bool near = lane < total && r2 < a.p.rcut * a.p.rcut && r2 > 0.0f && et >= 0 && et < NS;
    const unsigned long long below = (1ull << lane) - 1ull;
    int nn = 0, pos = 0;
    unsigned pairs = 0;                                  // number of the pair with type p at bits 4p, four times the own type from bit 20
#pragma unroll
    for (int e = 0; e < NS; ++e) {
        const unsigned long long mask = __ballot(near && et == e);
        if (et == e) {
            unsigned w = 4u * e << 20;
#pragma unroll
            for (int p = 0; p < NS; ++p) {
                const int lo = p < e ? p : e, hi = p < e ? e : p;
                w |= (unsigned)(lo * NS - lo * (lo - 1) / 2 + hi - lo) << (4 * p);
            }
            pairs = w;
            pos = nn + __popcll(mask & below);
        }
        nn += __popcll(mask);
    }
    if (near && wave == 0) {
        const float ir = __builtin_amdgcn_rsqf(r2), r = root(r2, ir);
        float fc, dfc;
        cutoff(r, inv_rc, fc, dfc);
        reinterpret_cast<float4*>(recA)[pos] = make_float4(dx, dy, dz, r);
        reinterpret_cast<float4*>(recB)[pos] = make_float4(ir, fc, dfc, __uint_as_float(pairs));
        sj[pos] = lane;
    }
    // the incoming gradient, times the constant factor of its bin
    const float f3 = !bin_ok ? 0.0f : a.gscale * (even ? group_factor(ul, l3, lane, spacing) : 1.0f);
    if constexpr (!ONE) {
        gsrc = gradient();
        const float f2 = a.gscale * frcp(rs2v);
        if (wave == 0 && lane < 32) slnRs2[lane] = flog(rs2v);
        for (int e = 2 * wave + (lane >> 5); e < NS; e += 2 * NW) gin2[32 * e + z] = z < nRs2 ? gsrc[e * nRs2 + z] * f2 : 0.0f;
        for (int pq = 3 * wave + third; pq < NP; pq += 3 * NW) {
            float2 g = make_float2(0.f, 0.f);
            if (bin_ok) g = make_float2(gsrc[NS * nRs2 + 2 * (pq * nRs3 + l3)] * f3, gsrc[NS * nRs2 + 2 * (pq * nRs3 + l3) + 1] * f3);
            if (lane < STEP) reinterpret_cast<float2*>(gin3)[LEAN_RS3 * pq + l3] = g;
        }
    } else {
        const float f2 = a.gscale * frcp(rs2v);
        if (lane < 32) slnRs2[lane] = flog(rs2v);
#pragma unroll
        for (int k = 0; k < (NS + 1) / 2; ++k)
            if (64 * k + lane < 32 * NS) gin2[64 * k + lane] = g2[k] * f2;
#pragma unroll
        for (int k = 0; k < (NP + 2) / 3; ++k)
            if (lane < STEP && 3 * k + third < NP)
                reinterpret_cast<float2*>(gin3)[STEP * k + lane] = make_float2(g3[k].x * f3, g3[k].y * f3);
    }
    __syncthreads();
    const float4* rA = reinterpret_cast<const float4*>(recA);
    const float4* rB = reinterpret_cast<const float4*>(recB);
    float gix = 0.0f, giy = 0.0f, giz = 0.0f;

    // ---- two-body: lanes = (bin group, neighbour); see fchl19_vjp_kernel ----
    if (wave == 0) {
        const int G = nn > 0 ? idiv_small(64, nn) : 1;       // nn < 64
        const int g = G > 1 ? idiv_small(lane, nn) : 0, j = lane - g * nn;
        const bool active = g < G && j < nn;
        float gr = 0.0f;
        float4 Aj = make_float4(0.f, 0.f, 0.f, 1.f), Bj = make_float4(1.f, 0.f, 0.f, 0.f);
        if (active) {
            Aj = rA[j];
            Bj = rB[j];
            const TwoBody tb = two_body_setup(Aj.w, Bj.y, Bj.z, a.p);
            const float inv_s2 = frcp(tb.s2);
            const float nc = -0.5f * LOG2E * inv_s2;
            const float hs = 0.5f * tb.s2p * inv_s2;
            const float q0 = fmaf(tb.fc, -hs - tb.d2_over_r, tb.dfc);
            const float q1 = tb.fc * inv_s2 * tb.mup;
            const float q2 = tb.fc * hs * inv_s2;
            const float* gz = gin2 + (__float_as_uint(Bj.w) >> 22) * 32 + g;
            const float* lz = slnRs2 + g;
            for (int zz = g; zz < nRs2; zz += G, gz += G, lz += G) {
                const float u = *lz - tb.mu;
                const float e = fexp2(u * u * nc);
                gr = fmaf(*gz * e, fmaf(fmaf(q2, u, q1), u, q0), gr);
            }
            gr *= tb.pre;
        }
        float tot = gr;
        for (int k = 1; k < G; ++k) tot += __shfl(gr, (lane + nn * k) & 63, 64);
        if (active && g == 0) {
            const float ux = Aj.x * Bj.x, uy = Aj.y * Bj.x, uz = Aj.z * Bj.x;   // dr/dR_i
            gix = tot * ux;
            giy = tot * uy;
            giz = tot * uz;
            reinterpret_cast<float4*>(mine)[j] = make_float4(-tot * ux, -tot * uy, -tot * uz, 0.0f);
        }
    }
    if constexpr (ONE) __syncthreads();                  // (the others have copies of their own)

    // ---- three-body: lane = triple; see fchl19_vjp_kernel for the numbering, the copies and the formulas ----
    float us[LEAN_RS3], ratio[LEAN_RS3 / RS3_GROUP];     // the grid, on scalar registers
#pragma unroll
    for (int l = 0; l < LEAN_RS3; ++l) us[l] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ul), l));
    {
        const float v = group_ratio<0>(-spacing, ul);
#pragma unroll
        for (int q = 0; q < LEAN_RS3 / RS3_GROUP; ++q) ratio[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), RS3_GROUP * q));
    }
    const int ntrip = (nn * (nn - 1)) >> 1;
    const float zw3 = 0.014383766711652736f * a.p.three_body_weight;     // 2 exp(-pi^2 / 2)
    const float d3 = a.p.three_body_decay;
    const float inn = frcp((float)nn);
    auto add_force = [&](float* p, float x, float y, float z) {
        float4 f = *reinterpret_cast<float4*>(p);
        f.x += x;
        f.y += y;
        f.z += z;
        *reinterpret_cast<float4*>(p) = f;
    };
    for (int t0 = QMLL_WAVE * wave; t0 < ntrip; t0 += QMLL_WAVE * NW) {
        const int tt = t0 + lane;
        if (tt >= ntrip) break;
        const int s0 = __builtin_amdgcn_readfirstlane((int)(((float)t0 + 0.5f) * inn));
        const int s = (int)(((float)tt + 0.5f) * inn), j = tt - __mul24(s, nn);
        int k = j + s + 1;
        if (k >= nn) k -= nn;
        float* copy = mine + 4 * __mul24(s - s0, nn);
        const float4 Aj = rA[j], Ak = rA[k], Bj = rB[j], Bk = rB[k];
        const float ia = Bj.x, ib = Bk.x;
        const float cx = Ak.x - Aj.x, cy = Ak.y - Aj.y, cz = Ak.z - Aj.z;
        const float c2 = cx * cx + cy * cy + cz * cz;
        const float ic = __builtin_amdgcn_rsqf(c2), c = c2 * ic;
        const float vi = Aj.x * Ak.x + Aj.y * Ak.y + Aj.z * Ak.z;
        const float dac = Aj.x * cx + Aj.y * cy + Aj.z * cz;
        const float dcb = cx * Ak.x + cy * Ak.y + cz * Ak.z;
        const float w = ia * ib, iaic = ia * ic, ibic = ib * ic;
        const float ci = vi * w, cj = -dac * iaic, ck = dcb * ibic;
        // a^2 b^2 - (d_ij.d_ik)^2 = |d_ij x d_ik|^2 (Lagrange): the cross product keeps full
        // relative accuracy near collinear triples, where the difference of squares cancels
        const float px = Aj.y * Ak.z - Aj.z * Ak.y, py = Aj.z * Ak.x - Aj.x * Ak.z, pz = Aj.x * Ak.y - Aj.y * Ak.x;
        const float cross2 = px * px + py * py + pz * pz;
        const float cosT = fminf(1.0f, fmaxf(-1.0f, ci));
        const float sinT = fminf(1.0f, fsqrt(cross2) * w);
        const float guard_inv = Aj.w * Ak.w * __builtin_amdgcn_rsqf(fmaxf(1e-10f, cross2));
        const float q1 = cj * ck, q2 = ci * ck, q3 = ci * cj;
        const float X = ci * q1, X2 = X + X;
        const float P = fmaf(3.0f, X, 1.0f);
        const float Pa3 = fmaf(q1, ib, fmaf(q2, ic, fmaf(-q3 * Aj.w, ibic, -X2 * ia)));
        const float Pb3 = fmaf(q1, ia, fmaf(q3, ic, fmaf(-q2 * Ak.w, iaic, -X2 * ib)));
        const float Pc3 = fmaf(q2, ia, fmaf(q3, ib, fmaf(-q1 * c, w, -X2 * ic)));
        const float Z = zw3 * fexp2(-d3 * flog2(Aj.w * Ak.w * c));
        const float fa = Bj.y, dfa = Bj.z, fb = Bk.y, dfb = Bk.z;
        const float F = fa * fb, d3P = d3 * P, FP = F * P;
        const float ka = fmaf(F, fmaf(3.0f, Pa3, -d3P * ia), P * dfa * fb);   // K_a / dec
        const float kb = fmaf(F, fmaf(3.0f, Pb3, -d3P * ib), P * fa * dfb);
        const float kc = F * fmaf(3.0f, Pc3, -d3P * ic);
        // the bins of this triple's pair of types
        const unsigned pair = __builtin_amdgcn_ubfe(__float_as_uint(Bk.w), __float_as_uint(Bj.w) >> 20, 4);
        const float4* g = reinterpret_cast<const float4*>(gin3 + __mul24((int)pair, 2 * LEAN_RS3));
        const float y = fmaf(sk3 * 0.5f, Aj.w + Ak.w, -mid);
        float Gc = 0.f, Gs = 0.f, Hc = 0.f, Hs = 0.f;
        auto groups = [&](auto stop) {
            const float B = group_ratio<0>(spacing, y);
            const float2* g2 = reinterpret_cast<const float2*>(g);
#pragma unroll
            for (int q = 0; q < LEAN_RS3 / RS3_GROUP; ++q) {
                const float d = y - us[RS3_GROUP * q], Q = B * ratio[q];
                group_sums(g2 + RS3_GROUP * q, d, fexp2(-(d * d)), decltype(stop)::value ? fminf(Q, RATIO_STOP) : Q, spacing, Gc, Gs, Hc, Hs);
            }
        };
        if (__builtin_expect(even && !stops, 1)) {
            groups(std::false_type{});
        } else if (even) {
            groups(std::true_type{});
        } else {
            auto bin = [&](float gc, float gs, float u) {
                const float dl = y - u;
                const float e = fexp2(-(dl * dl));
                const float de = dl * e;
                Gc = fmaf(gc, e, Gc);
                Gs = fmaf(gs, e, Gs);
                Hc = fmaf(gc, de, Hc);
                Hs = fmaf(gs, de, Hs);
            };
#pragma unroll
            for (int l = 0; l < LEAN_RS3; l += 2) {
                const float4 gv = g[l / 2];
                bin(gv.x, gv.y, us[l]);
                bin(gv.z, gv.w, us[l + 1]);
            }
        }
        const float S0 = Gc * cosT + Gs * sinT;
        const float S1 = 0.5f * hfac * (Hc * cosT + Hs * sinT);                   // d rho/da = d rho/db = 1/2
        const float Sth = (Gc * sinT - Gs * cosT) * guard_inv;                     // multiplies d cos_i
        const float ea = Z * ia * fmaf(ka, S0, FP * fmaf(Sth, fmaf(-ci, ia, ib), S1));   // (d L / d a) / a
        const float eb = Z * ib * fmaf(kb, S0, FP * fmaf(Sth, fmaf(-ci, ib, ia), S1));
        const float ec = Z * ic * fmaf(kc, S0, -FP * Sth * c * w);
        gix = fmaf(ea, Aj.x, fmaf(eb, Ak.x, gix));
        giy = fmaf(ea, Aj.y, fmaf(eb, Ak.y, giy));
        giz = fmaf(ea, Aj.z, fmaf(eb, Ak.z, giz));
        add_force(copy + 4 * j, fmaf(ec, cx, -ea * Aj.x), fmaf(ec, cy, -ea * Aj.y), fmaf(ec, cz, -ea * Aj.z));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the next read sees every lane's write (LDS instructions run in order)
        add_force(copy + 4 * k, fmaf(-ec, cx, -eb * Ak.x), fmaf(-ec, cy, -eb * Ak.y), fmaf(-ec, cz, -eb * Ak.z));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if constexpr (ONE) __syncthreads();
    gix = wave_sum(gix);
    giy = wave_sum(giy);
    giz = wave_sum(giz);
    if constexpr (!ONE) {
        if (lane == 0) own_force[3 * wave] = gix, own_force[3 * wave + 1] = giy, own_force[3 * wave + 2] = giz;
        __syncthreads();
    }
    float* gm = grad_X + (size_t)m * a.n * 3;
    const int ncopies = force_copies(nn);
    const int busy = ONE ? 1 : min(NW, max(1, (ntrip + QMLL_WAVE - 1) / QMLL_WAVE));      // wavefronts that have had triples, or the two-body part
    for (int it = ONE ? lane : threadIdx.x; it < 3 * (nn + 1); it += QMLL_WAVE * NW) {
        const int x = idiv_small(it, 3), c = it - 3 * x;
        float sum = c == 0 ? gix : c == 1 ? giy : giz;   // on atom i itself
        int to = i;
        if (x < nn) {
            to = sj[x];
            sum = 0.0f;
            for (int w = 0; w < busy; ++w)
                for (int q = 0; q < ncopies; ++q) sum += force[4 * (w * a.tcap + q * nn + x) + c];
        } else if (!ONE) {
            sum = 0.0f;
            for (int w = 0; w < busy; ++w) sum += own_force[3 * w + c];
        }
        atomicAdd(&gm[to * 3 + c], sum);
    }
}

template <int NS>
__global__ __launch_bounds__(64) void fchl19_vjp_lean_kernel(FchlArgs a, const float* __restrict__ grad_rep, float* __restrict__ grad_X) {
    extern __shared__ float smem[];
    const int m = a.molIDs[blockIdx.x];
    const int i = a.atomIDs[blockIdx.x];
    if (m < 0 || m >= a.B || i < 0 || i >= a.n) return;   // malformed index: write nothing
    const int R = NS * a.p.nRs2 + NS * (NS + 1) * a.p.nRs3;
    lean_vjp<NS, 1>(a, m, i, smem, [&] { return grad_rep + ((size_t)m * a.n + i) * R; }, grad_X);
}

// The backward projection and the VJP of few atoms in one launch: a workgroup per atom (in sorted order) forms its row of the
// representation's gradient in LDS, g_rep = sum of the parts of gx . U^T, four lanes to an entry, and takes it from there.  Both
// were chains of latencies in launches of their own; here the reductor's rows are on their way while the neighbours are staged, and the
// triples are shared by eight wavefronts.  Workgroups behind the atoms sum the energies, a wavefront per molecule.  21 atoms, 128
// components: 4.1 + 7.2 us, 8.3 so.  With the forward pair (above) energies and forces of 1 x 21 atoms take 21.3 us (28.5), 12 x 21 25.4 (30.7),
// 8 x 29 26.0 (32.1), 20 x 12 at 64 components 21.0 (26.2).  Beyond 256 atoms the workgroups, a CU each, come in rounds: 16 x 21 41.7 (37.7); with rows
// read in several pieces (five elements or 256 components) the pieces wait for memory: 2 x 29, five elements, 128 components 34.4 (32.9).
struct ProjectedGradient {
    const float* gx;              // [nparts][A][d]
    int nparts;
    const int* sorted_slots;
    const int* type_offsets;
    const float* reductors;       // [ne][R][d]
    int ne, A;
    const float* e_slots;         // [nparts][B n]
    float* energies;              // or null
};
template <int NS, int D, int W>
__global__ __launch_bounds__(64 * W) void fchl19_projected_vjp_kernel(FchlArgs a, ProjectedGradient pg, float* __restrict__ grad_X) {
    extern __shared__ float smem[];
    constexpr int ROWS = 16 * W, KQ = D / 16, AHEAD = held_rows(D, W) / ROWS;
    const int tid = threadIdx.x, R = NS * a.p.nRs2 + NS * (NS + 1) * a.p.nRs3;
    const int pos = blockIdx.x;
    if (pos >= pg.A) {                                   // energies: a wavefront per molecule
        const int mol = (pos - pg.A) * W + (tid >> 6), lane = tid & 63;
        if (mol >= a.B) return;
        float acc = 0.0f;
        for (int t = lane; t < pg.nparts * a.n; t += 64) {
            const int part = t / a.n;
            acc += pg.e_slots[((size_t)part * a.B + mol) * a.n + (t - part * a.n)];
        }
        acc = wave_sum(acc);
        if (lane == 0) pg.energies[mol] = acc;
        return;
    }
    if (pos >= pg.type_offsets[pg.ne]) return;           // atoms of elements that the model does not know come last and have no gradient
    int e = 0;
    while (e + 1 < pg.ne && pos >= pg.type_offsets[e + 1]) ++e;
    const float* U = pg.reductors + (size_t)e * R * D;
    const int q = tid & 3, r0 = tid >> 2;
    float4 u[AHEAD][KQ];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
#pragma unroll
        for (int c = 0; c < KQ; ++c) {
            u[j][c] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (ROWS * j < R) u[j][c] = reinterpret_cast<const float4*>(U + (size_t)min(r0 + ROWS * j, R - 1) * D)[q + 4 * c];
        }
    float v = 0.0f;
    if (tid < D) {
        const float* g = pg.gx + (size_t)pos * D + tid;
#pragma unroll 12
        for (int k = 0; k < pg.nparts; ++k) v += g[(size_t)k * pg.A * D];
    }
    const int slot = pg.sorted_slots[pos], m = slot / a.n, i = slot - m * a.n;
    float* sg = smem;                                    // [D] gx
    float* row = sg + D;                                 // [R4] g_rep
    lean_vjp<NS, W>(a, m, i, row + ((R + 3) & ~3), [&]() -> const float* {
        if (tid < D) sg[tid] = v;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            if (ROWS * j >= R) break;
            float sum = 0.0f;
#pragma unroll
            for (int c = 0; c < KQ; ++c) {
                const float4 g = reinterpret_cast<const float4*>(sg)[q + 4 * c];
                sum = fmaf(u[j][c].x, g.x, fmaf(u[j][c].y, g.y, fmaf(u[j][c].z, g.z, fmaf(u[j][c].w, g.w, sum))));
            }
            sum += lane_xor<1>(sum);
            sum += lane_xor<2>(sum);
            if (q == 0 && r0 + ROWS * j < R) row[r0 + ROWS * j] = sum;
        }
        __syncthreads();
        return row;
    }, grad_X);
}

// ---------------------------------------------------------------------------------
// explicit Jacobian (and the representation itself when rep != NULL)
//
// Output-centric and atomic-free: the wavefront of central atom i produces, one target
// atom at a time (i itself, then each neighbour), the three rows jac[m,i,target,0..2,:]
// in an LDS row buffer and streams them out coalesced.  For a neighbour target only the
// triples that contain it contribute; for the self row all triples do.
// ---------------------------------------------------------------------------------
// TABLE: everything of a triple that does not depend on the radial bin (geometry, the partials of
// the angular and decay factors, the unit vectors) is computed once per triple into an LDS table
// of JT floats; the (triple, radial bin) items of every target pass then only read it.  Without
// the table each item recomputes its triple, nRs3 times over and again in the neighbour passes.
constexpr int JT = 20;   // rho, bin offset, 6 alpha, 2 beta, u_ij, u_ik, u_jk, pad
constexpr int JW_MOST = 4;       // wavefronts per central atom
template <bool TABLE>
__global__ __launch_bounds__(64 * JW_MOST) void fchl19_jacobian_kernel(FchlArgs a, float* __restrict__ rep,
                                                              float* __restrict__ jac, int all_rows) {
    extern __shared__ float smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    const int m = a.molIDs[blockIdx.x];
    const int i = a.atomIDs[blockIdx.x];
    if (m < 0 || m >= a.B || i < 0 || i >= a.n) return;   // malformed index: write nothing
    const int ns = a.p.nspecies, nRs2 = a.p.nRs2, nRs3 = a.p.nRs3;
    const int R = ns * nRs2 + ns * (ns + 1) * nRs3;

    Stage s = carve(smem, a.cap, ns);
    float* slnRs2 = s.next;          // [nRs2]
    float* sinvRs2 = slnRs2 + nRs2;  // [nRs2]
    float* sRs3 = sinvRs2 + nRs2;    // [nRs3]
    float* val = sRs3 + nRs3;        // [R]   representation row (self pass only)
    const int shared = nw > 1;
    int* next = reinterpret_cast<int*>(val + R);             // the next target (of several wavefronts)
    float* row = val + R + shared + wave * 3 * R;            // [3][R] rows that this wavefront assembles
    // TABLE: [ntrip][JT], 16-byte aligned behind the rows
    float* ttab = val + R + shared + 3 * R * nw;
    ttab += (4 - ((size_t)(ttab - smem) & 3)) & 3;

    for (int t = threadIdx.x; t < nRs2; t += blockDim.x) {
        const float v = a.Rs2[t];
        slnRs2[t] = flog(v);
        sinvRs2[t] = frcp(v);
    }
    for (int t = threadIdx.x; t < nRs3; t += blockDim.x) sRs3[t] = a.Rs3[t];
    if (shared && threadIdx.x == 0) *next = 0;
    // (every wavefront stages the same neighbours in the same places)
    const int nn = stage_neighbours(a, s, m, i, lane);
    __syncthreads();

    const float k3 = a.p.eta3 * LOG2E;
    const float zeta2 = 0.014383766711652736f;   // 2 exp(-pi^2 / 2)
    float* jbase = jac + (((size_t)m * a.n + i) * a.n) * 3 * R;

    if constexpr (TABLE) {
        // T_c = zeta2 K e cosT, T_s = zeta2 K e sinT with e = exp(-eta3 (rho - Rs_l)^2): their partials
        // with respect to the three distances are e * alpha + (de/drho) * beta, alpha and beta per triple
        const int ntrip = nn * (nn - 1) / 2;
        for (int tt = threadIdx.x; tt < ntrip; tt += blockDim.x) {
            int j, k;
            unrank_pair(tt, nn, j, k);
            const Triple t = triple_geometry(s, j, k);
            const TripleDeriv d = triple_derivatives(t, a.p, s.fc[j], s.dfc[j], s.fc[k], s.dfc[k]);
            const float dcos = t.sinT * t.guard_inv;       // d cosT = dcos * d cos_i
            const float dsin = -t.cosT * t.guard_inv;      // d sinT = dsin * d cos_i
            const float ia = frcp(t.a), ib = frcp(t.b);
            float4* e4 = reinterpret_cast<float4*>(ttab + (size_t)tt * JT);
            e4[0] = make_float4(0.5f * (t.a + t.b),
                                __int_as_float(pair_offset(s.el[j], s.el[k], ns, nRs2, nRs3)),
                                zeta2 * (d.Ka * t.cosT + d.K * dcos * d.cia),
                                zeta2 * (d.Kb * t.cosT + d.K * dcos * d.cib));
            e4[1] = make_float4(zeta2 * (d.Kc * t.cosT + d.K * dcos * d.cic),
                                zeta2 * (d.Ka * t.sinT + d.K * dsin * d.cia),
                                zeta2 * (d.Kb * t.sinT + d.K * dsin * d.cib),
                                zeta2 * (d.Kc * t.sinT + d.K * dsin * d.cic));
            e4[2] = make_float4(zeta2 * d.K * t.cosT, zeta2 * d.K * t.sinT, s.dx[j] * ia, s.dy[j] * ia);
            e4[3] = make_float4(s.dz[j] * ia, s.dx[k] * ib, s.dy[k] * ib, s.dz[k] * ib);
            e4[4] = make_float4(t.ujk[0], t.ujk[1], t.ujk[2], 0.0f);
        }
        __syncthreads();
    }

    // target = -1: central atom; target = 0..nn-1: neighbour at that list position.  Each wavefront takes the next one that is left,
    // and the rows of its own: nothing below waits for another wavefront
    for (int target = -1;; ++target) {
        if (shared) {
            int taken = 0;
            if (lane == 0) taken = atomicAdd(next, 1);
            target = __builtin_amdgcn_readfirstlane(taken) - 1;
        }
        if (target >= nn) {
            // (all rows: then those of the atoms that are no target, three rows of zeros each)
            const int j = target - nn;
            if (!all_rows || j >= a.n) break;
            bool seen = j == i;
            for (int k = lane; k < nn; k += QMLL_WAVE) seen |= s.j[k] == j;
            if (!__any(seen))
                for (int t = lane; t < 3 * R; t += QMLL_WAVE) jbase[(size_t)j * 3 * R + t] = 0.0f;
            continue;
        }
        for (int t = lane; t < 3 * R; t += QMLL_WAVE) row[t] = 0.0f;
        if (target < 0)
            for (int t = lane; t < R; t += QMLL_WAVE) val[t] = 0.0f;
        wave_sync();

        // two-body: items (neighbour j, bin z); a neighbour target only sees its own pair
        {
            const int j0 = target < 0 ? 0 : target;
            const int j1 = target < 0 ? nn : target + 1;
            const float sign = target < 0 ? 1.0f : -1.0f;   // dr/dR_i = u_ij, dr/dR_j = -u_ij
            for (int it = lane; it < (j1 - j0) * nRs2; it += QMLL_WAVE) {
                const int jq = idiv_small(it, nRs2);
                const int j = j0 + jq;
                const int z = it - jq * nRs2;
                const float r = s.r[j];
                const TwoBody tb = two_body_setup(r, s.fc[j], s.dfc[j], a.p);
                float v, dv;
                two_body_bin(tb, slnRs2[z], sinvRs2[z], v, dv);
                const float ir = sign * dv * frcp(r);
                const int bin = s.el[j] * nRs2 + z;
                atomicAdd(&row[0 * R + bin], ir * s.dx[j]);
                atomicAdd(&row[1 * R + bin], ir * s.dy[j]);
                atomicAdd(&row[2 * R + bin], ir * s.dz[j]);
                if (target < 0) atomicAdd(&val[bin], v);
            }
        }
        // three-body with the table: owner computes.  Lanes = (triple sub-slot, radial bin l); a lane
        // sums its bin over the triples of one element pair in registers (no LDS atomics, which run
        // at one lane per clock), sub-slots are folded with shuffles, sub-slot 0 stores the bin.
        if constexpr (TABLE) {
            const int W3 = nRs3 < 64 ? nRs3 : 64;
            const int TS = idiv_small(64, W3);
            const int tsub = idiv_small(lane, W3), ll = lane - tsub * W3;
            // the triples of one block: index it -> neighbour positions j < k
            auto block = [&](int off_pair, int count, int p, int q) {
                const int op = s.goff[p], oq = s.goff[q];
                const int np_ = s.goff[p + 1] - op, nq = s.goff[q + 1] - oq;
                for (int lb = 0; lb * 64 < nRs3; ++lb) {
                    const int l = lb * 64 + ll;
                    const bool lok = l < nRs3 && tsub < TS;
                    const float rs = sRs3[lok ? l : 0];
                    float gc[3] = {0.f, 0.f, 0.f}, gs[3] = {0.f, 0.f, 0.f}, vc = 0.f, vs = 0.f;
                    for (int it = tsub; it < count && lok; it += TS) {
                        int j, k;
                        if (target < 0) {
                            if (p == q) {
                                unrank_pair(it, np_, j, k);
                                j += op;
                                k += op;
                            } else {
                                j = op + it / nq;
                                k = oq + it - (it / nq) * nq;
                            }
                        } else {   // q is the element of the other neighbour o; p that of the target
                            int o = oq + it;
                            if (p == q && o >= target) ++o;
                            j = o < target ? o : target;
                            k = o < target ? target : o;
                        }
                        const float4* e4 = reinterpret_cast<const float4*>(
                            ttab + (size_t)((j * (2 * nn - j - 1)) / 2 + (k - j - 1)) * JT);
                        const float4 q0 = e4[0], q1 = e4[1], q2 = e4[2], q3 = e4[3], q4 = e4[4];
                        const float dl = q0.x - rs;
                        const float e = fexp2(-k3 * dl * dl);
                        const float de = -a.p.eta3 * dl * e;      // (d e/d rho) * (d rho/d a)
                        const float Tca = fmaf(e, q0.z, de * q2.x), Tcb = fmaf(e, q0.w, de * q2.x), Tcc = e * q1.x;
                        const float Tsa = fmaf(e, q1.y, de * q2.y), Tsb = fmaf(e, q1.z, de * q2.y), Tsc = e * q1.w;
                        const float ua[3] = {q2.z, q2.w, q3.x};
                        const float ub[3] = {q3.y, q3.z, q3.w};
                        const float uc[3] = {q4.x, q4.y, q4.z};
                        if (target < 0) {            // d/dR_i, and the value itself
                            vc = fmaf(e, q2.x, vc);
                            vs = fmaf(e, q2.y, vs);
#pragma unroll
                            for (int x = 0; x < 3; ++x) {
                                gc[x] += Tca * ua[x] + Tcb * ub[x];
                                gs[x] += Tsa * ua[x] + Tsb * ub[x];
                            }
                        } else if (j == target) {    // d/dR_j
#pragma unroll
                            for (int x = 0; x < 3; ++x) {
                                gc[x] += -Tca * ua[x] + Tcc * uc[x];
                                gs[x] += -Tsa * ua[x] + Tsc * uc[x];
                            }
                        } else {                     // d/dR_k
#pragma unroll
                            for (int x = 0; x < 3; ++x) {
                                gc[x] += -Tcb * ub[x] - Tcc * uc[x];
                                gs[x] += -Tsb * ub[x] - Tsc * uc[x];
                            }
                        }
                    }
                    // fold the sub-slots: totals apart from the partial sums the other lanes read
                    float tc[3] = {gc[0], gc[1], gc[2]}, tsn[3] = {gs[0], gs[1], gs[2]}, tvc = vc, tvs = vs;
                    for (int kk = 1; kk < TS; ++kk) {
                        const int src = ll + W3 * kk;
#pragma unroll
                        for (int x = 0; x < 3; ++x) {
                            tc[x] += __shfl(gc[x], src, 64);
                            tsn[x] += __shfl(gs[x], src, 64);
                        }
                        tvc += __shfl(vc, src, 64);
                        tvs += __shfl(vs, src, 64);
                    }
                    if (tsub == 0 && l < nRs3) {
                        const int off = off_pair + 2 * l;
#pragma unroll
                        for (int x = 0; x < 3; ++x) {
                            row[x * R + off] = tc[x];
                            row[x * R + off + 1] = tsn[x];
                        }
                        if (target < 0) {
                            val[off] = tvc;
                            val[off + 1] = tvs;
                        }
                    }
                }
            };
            if (target < 0) {
                for (int p = 0; p < ns; ++p) {
                    const int np_ = s.goff[p + 1] - s.goff[p];
                    for (int q = p; q < ns; ++q) {
                        const int nq = s.goff[q + 1] - s.goff[q];
                        block(pair_offset(p, q, ns, nRs2, nRs3), p == q ? np_ * (np_ - 1) / 2 : np_ * nq, p, q);
                    }
                }
            } else {
                const int p = s.el[target];
                for (int q = 0; q < ns; ++q) {
                    const int nq = s.goff[q + 1] - s.goff[q];
                    block(pair_offset(p, q, ns, nRs2, nRs3), nq - (p == q ? 1 : 0), p, q);
                }
            }
        } else {
            // self: all pairs (j<k); neighbour target: the nn-1 pairs {target, other}
            const int ntr = target < 0 ? nn * (nn - 1) / 2 : nn - 1;
            for (int it = lane; it < ntr * nRs3; it += QMLL_WAVE) {
                const int tt = idiv_small(it, nRs3);
                const int l = it - tt * nRs3;
                int j, k;
                if (target < 0) {
                    unrank_pair(tt, nn, j, k);
                } else {
                    const int o = tt < target ? tt : tt + 1;
                    j = o < target ? o : target;
                    k = o < target ? target : o;
                }
                const Triple t = triple_geometry(s, j, k);
                const TripleDeriv d = triple_derivatives(t, a.p, s.fc[j], s.dfc[j], s.fc[k], s.dfc[k]);
                const float rho = 0.5f * (t.a + t.b);
                const float dl = rho - sRs3[l];
                const float e = fexp2(-k3 * dl * dl);
                const float de = -a.p.eta3 * dl * e;          // (d e/d rho) * (d rho/d a)
                // T_c = zeta2 K e cosT, T_s = zeta2 K e sinT; partials wrt a, b, c
                const float dcos = t.sinT * t.guard_inv;       // d cosT = dcos * d cos_i
                const float dsin = -t.cosT * t.guard_inv;      // d sinT = dsin * d cos_i
                float Tca, Tcb, Tcc, Tsa, Tsb, Tsc;
                {
                    const float Ke = zeta2 * d.K * e;
                    const float base_a = zeta2 * (d.Ka * e + d.K * de);
                    const float base_b = zeta2 * (d.Kb * e + d.K * de);
                    const float base_c = zeta2 * (d.Kc * e);
                    Tca = base_a * t.cosT + Ke * dcos * d.cia;
                    Tcb = base_b * t.cosT + Ke * dcos * d.cib;
                    Tcc = base_c * t.cosT + Ke * dcos * d.cic;
                    Tsa = base_a * t.sinT + Ke * dsin * d.cia;
                    Tsb = base_b * t.sinT + Ke * dsin * d.cib;
                    Tsc = base_c * t.sinT + Ke * dsin * d.cic;
                    if (target < 0) {
                        const int off = pair_offset(s.el[j], s.el[k], ns, nRs2, nRs3) + 2 * l;
                        atomicAdd(&val[off], Ke * t.cosT);
                        atomicAdd(&val[off + 1], Ke * t.sinT);
                    }
                }
                const float ia = frcp(t.a), ib = frcp(t.b);
                const float ua[3] = {s.dx[j] * ia, s.dy[j] * ia, s.dz[j] * ia};
                const float ub[3] = {s.dx[k] * ib, s.dy[k] * ib, s.dz[k] * ib};
                const int off = pair_offset(s.el[j], s.el[k], ns, nRs2, nRs3) + 2 * l;
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    float gc, gs;
                    if (target < 0) {            // d/dR_i
                        gc = Tca * ua[x] + Tcb * ub[x];
                        gs = Tsa * ua[x] + Tsb * ub[x];
                    } else if (j == target) {    // d/dR_j
                        gc = -Tca * ua[x] + Tcc * t.ujk[x];
                        gs = -Tsa * ua[x] + Tsc * t.ujk[x];
                    } else {                     // d/dR_k
                        gc = -Tcb * ub[x] - Tcc * t.ujk[x];
                        gs = -Tsb * ub[x] - Tsc * t.ujk[x];
                    }
                    atomicAdd(&row[x * R + off], gc);
                    atomicAdd(&row[x * R + off + 1], gs);
                }
            }
        }
        wave_sync();
        const int tj = target < 0 ? i : s.j[target];
        float* dst = jbase + (size_t)tj * 3 * R;
        for (int t = lane; t < 3 * R; t += QMLL_WAVE) dst[t] = row[t];
        if (target < 0 && rep != nullptr) {
            float* out = rep + ((size_t)m * a.n + i) * R;
            for (int t = lane; t < R; t += QMLL_WAVE) out[t] = val[t];
        }
        wave_sync();
    }
}

int fill_args(FchlArgs& a, const float* X, const int* types, const float* cell, const float* inv_cell,
              const int* atomIDs, const int* molIDs, const int* natoms, const int* nlist, const int* nneigh,
              int nn_stride, int A, int B, int n, const float* Rs2, const float* Rs3, const qmll_fchl_params* prm,
              const char* who) {
    QMLL_REQUIRE(prm != nullptr, QMLL_ERR_INVALID, "%s: null params", who);
    QMLL_REQUIRE(A >= 0 && B >= 0 && n >= 0, QMLL_ERR_INVALID, "%s: negative size A=%d B=%d n=%d", who, A, B, n);
    QMLL_REQUIRE(prm->nspecies > 0 && prm->nRs2 > 0 && prm->nRs3 > 0, QMLL_ERR_INVALID,
                 "%s: nspecies=%d nRs2=%d nRs3=%d must be positive", who, prm->nspecies, prm->nRs2, prm->nRs3);
    QMLL_REQUIRE(prm->rcut > 0.0f, QMLL_ERR_INVALID, "%s: rcut must be positive", who);
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(X && types && atomIDs && molIDs && natoms && Rs2 && Rs3, QMLL_ERR_INVALID, "%s: null pointer", who);
    QMLL_REQUIRE((cell == nullptr) == (inv_cell == nullptr), QMLL_ERR_INVALID,
                 "%s: cell and inv_cell must both be given or both be NULL", who);
    QMLL_REQUIRE((nlist == nullptr) == (nneigh == nullptr), QMLL_ERR_INVALID,
                 "%s: nlist and nneigh must both be given or both be NULL", who);
    QMLL_REQUIRE(nlist == nullptr || nn_stride > 0, QMLL_ERR_INVALID, "%s: nn_stride=%d", who, nn_stride);
    a.X = X;
    a.types = types;
    a.cell = cell;
    a.inv_cell = inv_cell;
    a.atomIDs = atomIDs;
    a.molIDs = molIDs;
    a.natoms = natoms;
    a.nlist = nlist;
    a.nneigh = nneigh;
    a.nn_stride = nn_stride;
    a.n = n;
    a.B = B;
    a.cap = nlist ? nn_stride : n;
    if (a.cap < 1) a.cap = 1;
    a.tcap = 0;
    a.Rs2 = Rs2;
    a.Rs3 = Rs3;
    a.p = *prm;
    a.gscale = 1.0f;
    return QMLL_OK;
}

constexpr size_t LDS_LIMIT = 64 * 1024;

// Wavefronts per central atom.  With one, a launch of A atoms is A wavefronts: below about 1000 the chip (8192 slots at eight
// per SIMD) is idle while every atom walks through its phases alone, the longer the more triples it has; beyond, the work that
// every wavefront of an atom repeats (staging, the scan of the pairs) costs more than the idle slots, and the backward kernel, which
// also sums the wavefronts' forces, meets that with few triples at any A.  Measured, us per launch at three elements:
//   atoms x molecules (triples of an atom)   forward 1 / 4 / 8      backward 1 / 2 / 4
//   3 x 1 (1), 3 x 300                       6.1 / 5.8 / 5.9, 6.7 / 7.5 / 11.5        7.4 / 7.6 / 7.7, 8.3 / 8.5 / 9.5
//   12 x 1 (55), 12 x 20, 12 x 40, 12 x 90   7.6 / 7.0 / 6.9, 7.7 / 7.5 / 7.4, 8.0 / 7.9 / 8.3, 8.7 / 9.7 / 14.6
//                                                                   6.6 / 6.9 / 7.3, 6.7 / 6.9 / 7.4, 6.9 / 7.2 / 7.8, 7.4 / 8.0 / 9.9
//   21 x 1 (190), 21 x 12, 21 x 24, 21 x 48  9.4 / 7.6 / 7.3, 9.5 / 8.1 / 7.8, 10.0 / 8.8 / 8.9, 10.4 / 10.0 / 15.2
//                                                                   8.7 / 8.0 / 7.5, 9.0 / 8.1 / 7.8, 9.3 / 8.8 / 8.4, 9.3 / 9.0 / 10.1
//   29 x 8 (378), 29 x 20, 29 x 40           15.0 / 8.6 / 8.3, 15.8 / 9.9 / 10.8, 17.0 / 12.1 / 16.8
//                                                                   12.5 / 9.9 / 9.5, 13.2 / 11.1 / 10.9, 14.9 / 12.8 / 14.1
//   40 x 40 in a box                         25.8 / 18.6 / 25.4     23.9 / 23.1 / 24.1
//   96 x 2 in a box, 96 x 16                 78 / 29 / 23, 89 / 48 / 65               66 / 38 / 26, 86 / 65 / 54
// and at five elements 12 x 40: forward 11.9 / 10.5 / 10.4, 21 x 48: 14.7 / 13.5 / 18.5 and 10.0 / 9.7 / 10.4.  2016 atoms of 21: 11.7 / 16.6 and
// 11.3 / 16.6 with 1 / 4.
// big: the neighbourhood does not fit the one-wavefront kernel, or leaves it few wavefronts per CU.
// The kernels for a known number of elements (`lean`) do with fewer instructions per phase, so that one wavefront is the better choice
// up to some thirty atoms however few there are (us, 1 / 4 / 8 forward, 1 / 4 backward, three elements):
//   12 x 1, 12 x 40           4.4 / 6.8 / 7.0, 5.0 / 8.0 / 8.4          5.0 / 7.0, 5.4 / 7.7
//   21 x 1, 21 x 12, 21 x 48  5.9 / 7.7 / 7.5, 6.1 / 8.1 / 7.8, 6.8 / 10.0 / 14.3        7.0 / 7.4, 7.2 / 7.7, 7.6 / 10.2
//   29 x 1, 29 x 20 (four elements)     8.6 / 9.7 / 9.0, 9.7 / 11.7 / 12.5              10.3 / 9.0, 10.8 / 11.1
//   32 x 8 (465), 32 x 32     9.1 / 9.0 / 8.3, 10.3 / 11.6 / 16.3       11.3 / 9.2, 11.9 / 13.4
//   40 x 6 (741), 40 x 25, 40 x 50      11.9 / 10.1 / 8.9, 13.3 / 13.2 / 18.4, 15.5 / 21.8 / 27.6    15.0 / 10.4, 15.9 / 15.4, 21.0 / 23.9
//   46 x 6 (990), 46 x 22, 46 x 45      15.4 / 13.0 / 12.9, 16.1 / 16.5 / 23.4, 22.4 / 27.6 / 38.1   18.7 / 11.2, 19.4 / 17.2, 31.2 / 28.2
int wavefronts_forward(int A, long long triples, bool big, bool lean) {
    if (lean && !big) return triples <= 420 ? 1 : A <= 256 ? 8 : triples > 600 && A <= 768 ? 4 : 1;
    if (A <= 256) return 8;
    if (A <= (triples > 256 ? 2048 : triples > 100 ? 1024 : triples > 30 ? 512 : 256)) return 4;
    return big ? 4 : 1;
}
int wavefronts_backward(int A, long long triples, bool big, bool lean) {
    if (lean && !big) return A <= (triples > 900 ? 2048 : triples > 600 ? 1024 : triples > 256 ? 512 : 0) ? 4 : 1;
    if (A <= (triples > 256 ? 2048 : triples > 100 ? 768 : 0)) return 4;
    return big ? 4 : 1;
}

bool usual_bins(const qmll_fchl_params* prm) { return prm->nRs3 <= LEAN_RS3 && prm->nRs3 > LEAN_RS3 - 4; }

// What the kernels for a known number of elements take: five, because a place in the triple list has 11 bits of a 64-bit record; one
// candidate per lane; two-body bins on half a wavefront; and three-body bins that fill at least 17 of the 20 they are laid out
// for, where the general kernels have three sub-slots as well (with 16 they have four).
bool lean_grids(const qmll_fchl_params* prm, const int* nlist, int n) {
    return nlist == nullptr && prm->nspecies <= 5 && n <= QMLL_WAVE && prm->nRs2 <= 32 && usual_bins(prm);
}

}  // namespace

static int forward(const float* X, const int* types, const float* cell, const float* inv_cell, const int* atomIDs, const int* molIDs,
                   const int* natoms, const int* nlist, const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2,
                   const float* Rs3, const qmll_fchl_params* prm, const BatchPrep& prep, float* rep, qmll_stream_t stream) {
    FchlArgs a;
    int rc = fill_args(a, X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2, Rs3,
                       prm, "qmll_fchl19_forward");
    if (rc) return rc;
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(rep != nullptr, QMLL_ERR_INVALID, "qmll_fchl19_forward: null output");
    QMLL_REQUIRE(prm->nRs3 <= 256, QMLL_ERR_INVALID,
                 "qmll_fchl19_forward: nRs3=%d: at most 256 three-body radial bins are supported", prm->nRs3);
    const int R = prm->nspecies * prm->nRs2 + prm->nspecies * (prm->nspecies + 1) * prm->nRs3;
    // an atom has at most cap neighbours from a given list and at most max_atoms - 1 otherwise
    const long long maxnn = nlist ? a.cap : (a.cap > 1 ? a.cap - 1 : 1);
    const long long alltrip = maxnn * (maxnn - 1) / 2 > 0 ? maxnn * (maxnn - 1) / 2 : 1;
    const int ns = prm->nspecies, np = ns * (ns + 1) / 2;
    hipStream_t st = (hipStream_t)stream;
    const bool big = alltrip > TCH_MAX;
    for (int nw = wavefronts_forward(A, alltrip, big, lean_grids(prm, nlist, n)); nw > 1 || big; nw /= 2) {
        // the table holds the triple list, or 12 KB of it at a time
        a.tcap = alltrip <= TCH_WIDE ? (int)alltrip : TCH_WIDE;
        size_t lds = sizeof(float) * (4 * (size_t)(a.tcap + 1) + 12 * (size_t)a.cap + ns + 1 + 2 * prm->nRs2 + prm->nRs3 + np + 1 +
                                      (size_t)ns * nw + (nw > 1 ? (size_t)np * nw * 2 * prm->nRs3 : 0));
        if (nw == 1 && lds > LDS_LIMIT) {      // room for the neighbours of a large capacity: smaller pieces of the list
            const size_t less = std::min((lds - LDS_LIMIT + 15) / 16, (size_t)std::max(a.tcap - TCH_LEAST, 0));
            a.tcap -= (int)less;
            lds -= 16 * less;
        }
        if (lds > LDS_LIMIT) {          // many elements with fine grids: fewer wavefronts, fewer partial blocks
            QMLL_REQUIRE(nw > 1 || !big, QMLL_ERR_INVALID,
                         "qmll_fchl19_forward: %zu B of LDS needed (max_atoms=%d, repsize=%d) exceeds %zu", lds, n, R, LDS_LIMIT);
            continue;
        }
        const bool lean = usual_bins(prm);
        if (nw == 8 && lean) hipLaunchKernelGGL((fchl19_forward_wide_kernel<8, true>), dim3(A), dim3(512), lds, st, a, rep);
        else if (nw == 4 && lean) hipLaunchKernelGGL((fchl19_forward_wide_kernel<4, true>), dim3(A), dim3(256), lds, st, a, rep);
        else if (nw == 8) hipLaunchKernelGGL((fchl19_forward_wide_kernel<8, false>), dim3(A), dim3(512), lds, st, a, rep);
        else if (nw == 4) hipLaunchKernelGGL((fchl19_forward_wide_kernel<4, false>), dim3(A), dim3(256), lds, st, a, rep);
        else if (nw == 2) hipLaunchKernelGGL((fchl19_forward_wide_kernel<2, false>), dim3(A), dim3(128), lds, st, a, rep);
        else hipLaunchKernelGGL((fchl19_forward_wide_kernel<1, false>), dim3(A), dim3(64), lds, st, a, rep);
        QMLL_CHECK_LAUNCH("qmll_fchl19_forward");
        return QMLL_OK;
    }
    if (lean_grids(prm, nlist, n)) {
        const size_t entries = std::max<size_t>(alltrip + np * (LEAN_SLOTS - 1), a.cap);
        size_t lds = sizeof(float) * ((size_t)8 * a.cap + (3 * entries + 3) / 4 * 4);
        if (prep.Z) lds = std::max(lds, sizeof(int) * (size_t)A);        // the sort's
        auto launch = [&](auto nsc) {
            constexpr int NS = decltype(nsc)::value;
            if (prep.Z) hipLaunchKernelGGL((fchl19_forward_lean_kernel<NS, true>), dim3(prep.groups + A), dim3(64), lds, st, a, prep, rep);
            else hipLaunchKernelGGL((fchl19_forward_lean_kernel<NS, false>), dim3(A), dim3(64), lds, st, a, prep, rep);
        };
        switch (ns) {
            case 1: launch(std::integral_constant<int, 1>{}); break;
            case 2: launch(std::integral_constant<int, 2>{}); break;
            case 3: launch(std::integral_constant<int, 3>{}); break;
            case 4: launch(std::integral_constant<int, 4>{}); break;
            default: launch(std::integral_constant<int, 5>{}); break;
        }
        QMLL_CHECK_LAUNCH("qmll_fchl19_forward");
        return QMLL_OK;
    }
    // one wavefront per atom: two per-neighbour records [cap][4], type offsets, the radial grids, the pairs' segment starts,
    // and a table of as many triples as FORWARD_LDS leaves room for
    const size_t rest = sizeof(float) * ((size_t)8 * a.cap + ns + 1 + 2 * prm->nRs2 + prm->nRs3 + np + 1);
    const long long room = rest < FORWARD_LDS ? (long long)(FORWARD_LDS - rest) / 16 : 0;
    // each pair's part of the list is padded to a multiple of the triple sub-slot count, and so is the table
    const int unit = prm->nRs3 < 64 ? 64 / prm->nRs3 : 1;
    a.tcap = (int)std::max<long long>(std::min(alltrip + np * (unit - 1), std::max(room - unit, 128LL)), a.cap);
    a.tcap = (a.tcap + unit - 1) / unit * unit;
    const int least = (a.cap + unit - 1) / unit * unit;          // the two-body factors of the neighbours lie there first
    while (a.tcap > least && rest + 16 * (size_t)a.tcap > LDS_LIMIT) a.tcap -= unit;
    const size_t lds = rest + 16 * (size_t)a.tcap;
    QMLL_REQUIRE(lds <= LDS_LIMIT, QMLL_ERR_INVALID,
                 "qmll_fchl19_forward: %zu B of LDS needed (max_atoms=%d, repsize=%d) exceeds %zu", lds, n, R, LDS_LIMIT);
    hipLaunchKernelGGL(fchl19_forward_kernel, dim3(A), dim3(64), lds, st, a, rep);
    QMLL_CHECK_LAUNCH("qmll_fchl19_forward");
    return QMLL_OK;
}

extern "C" int qmll_fchl19_forward(const float* X, const int* types, const float* cell, const float* inv_cell,
                                   const int* atomIDs, const int* molIDs, const int* natoms, const int* nlist,
                                   const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2,
                                   const float* Rs3, const qmll_fchl_params* prm, float* rep, qmll_stream_t stream) {
    return forward(X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2, Rs3, prm, BatchPrep{}, rep,
                   stream);
}

// Where the batch can be prepared beside the representation.  One launch less and the bookkeeping beside the representation instead of ahead
// of it, where one wavefront does the sort before the atoms are done: energies and forces of 21 atoms 29.0 -> 26.0 us, 12 x 21 32.6 -> 29.4,
// 16 x 29 46.2 -> 43.3, but 42 x 12 (504 atoms) 29.0 -> 29.8 and 100 x 12 37.4 -> 45.3.
static bool prepared_beside(int A, long long slots, size_t zero_count, int ne, int n, const qmll_fchl_params* prm) {
    const long long maxnn = n > 1 ? n - 1 : 1, triples = maxnn * (maxnn - 1) / 2;
    return A > 0 && A <= PREP_ATOMS && slots > 0 && slots <= 32 * PREP_ATOMS && zero_count <= 128 * PREP_ATOMS && ne > 0 && ne <= PREP_ELEMENTS &&
           lean_grids(prm, nullptr, n) && wavefronts_forward(A, triples, triples > TCH_MAX, true) == 1;
}
static BatchPrep prep_of(const float* Z, const float* species, const float* model_species, int ne, int A, long long slots, int* types,
                         int* sort_types, int* sorted_slots, int* type_offsets, float* zero, size_t zero_count) {
    const long long work = std::max<long long>(slots, (long long)zero_count);
    return BatchPrep{Z, species, model_species, ne, A, (int)slots, types, sort_types, sorted_slots, type_offsets, zero, (int)zero_count,
                     1 + (int)((work + 255) / 256)};
}

extern "C" int qmll_prepare_fchl19_forward(const float* X, const float* Z, const float* species, const float* model_species, int ne,
                                           const float* cell, const float* inv_cell, const int* atomIDs, const int* molIDs,
                                           const int* natoms, int A, int B, int n, const float* Rs2, const float* Rs3,
                                           const qmll_fchl_params* prm, void* workspace, size_t workspace_bytes, int* types,
                                           int* sort_types, int* sorted_slots, int* type_offsets, float* zero, size_t zero_count,
                                           float* rep, qmll_stream_t stream) {
    QMLL_REQUIRE(prm != nullptr, QMLL_ERR_INVALID, "qmll_prepare_fchl19_forward: null params");
    const long long slots = (long long)B * n;
    BatchPrep b{};
    if (prepared_beside(A, slots, zero_count, ne, n, prm) && (model_species ? sort_types != nullptr : ne == prm->nspecies) && Z && species &&
        types && sorted_slots && type_offsets && (zero || zero_count == 0)) {
        b = prep_of(Z, species, model_species, ne, A, slots, types, sort_types, sorted_slots, type_offsets, zero, zero_count);
    } else {
        int rc = qmll_prepare_batch(Z, natoms, species, prm->nspecies, model_species, ne, atomIDs, molIDs, B, n, A, workspace,
                                    workspace_bytes, types, sort_types, sorted_slots, type_offsets, zero, zero_count, stream);
        if (rc != QMLL_OK) return rc;
    }
    return forward(X, types, cell, inv_cell, atomIDs, molIDs, natoms, nullptr, nullptr, 0, A, B, n, Rs2, Rs3, prm, b, rep, stream);
}

// Wavefronts per atom of the launches that take the projections in, 0: not taken.  Up to 256 atoms eight, a CU to each workgroup.  With
// more, two or four if they hold the reductor, and as many atoms as are resident at a time (twelve wavefronts per CU).  Energies and forces,
// 64 components, launches apart / so, us: two elements (two wavefronts) 300 atoms of 12 29.7 / 26.1, 1200 29.7 / 27.5, 1992 31.0 / 36.4; three
// elements (four) 492 29.4 / 26.7, 792 29.6 / 34.4; 100 x 12 through autograd 117 / 110.  Larger molecules too, also where the backward launch by
// itself would have four wavefronts an atom: two elements 33 atoms 495 32.4 / 28.8, 1485 39.0 / 34.6; 38 atoms 798 37.5 / 32.2, 1482 44.8 / 37.6; 46
// atoms 782 43.5 / 39.0, 1472 50.3 / 43.0; one element, 128 components, 46 atoms 1196 48.5 / 43.0; three elements, 36 atoms 756 40.4 / 32.9.  Only
// where the representation is the work of one wavefront: 3 x 40 atoms, 128 components, backward alone 31.9 / 32.9.
static int projected_waves(int A, int n, const qmll_fchl_params* prm, int d) {
    const int R = prm->nspecies * prm->nRs2 + prm->nspecies * (prm->nspecies + 1) * prm->nRs3;
    const long long maxnn = n > 1 ? n - 1 : 1, triples = maxnn * (maxnn - 1) / 2;
    if (A <= 0 || (d != 64 && d != 128) || !lean_grids(prm, nullptr, n) || wavefronts_forward(A, triples, triples > TCH_MAX, true) != 1) return 0;
    if (A <= PREP_ATOMS) return R <= held_rows(d, 8) ? 8 : 0;
    if (R <= held_rows(d, 2)) return A <= 6 * 256 ? 2 : 0;
    return R <= held_rows(d, 4) && A <= 3 * 256 ? 4 : 0;
}
// f(number of species, components, wavefronts) as constants, for what there can be
template <class F>
static void with_projected_shape(int ns, int d, int waves, F f) {
    auto by_waves = [&](auto nsc, auto dc) {
        constexpr int NS = decltype(nsc)::value, D = decltype(dc)::value;
        if constexpr (fewest_rows(NS) <= held_rows(D, 2)) {
            if (waves == 2) f(nsc, dc, std::integral_constant<int, 2>{});
        }
        if constexpr (fewest_rows(NS) <= held_rows(D, 4)) {
            if (waves == 4) f(nsc, dc, std::integral_constant<int, 4>{});
        }
        if (waves == 8) f(nsc, dc, std::integral_constant<int, 8>{});
    };
    auto by_species = [&](auto dc) {
        switch (ns) {
            case 1: by_waves(std::integral_constant<int, 1>{}, dc); break;
            case 2: by_waves(std::integral_constant<int, 2>{}, dc); break;
            case 3: by_waves(std::integral_constant<int, 3>{}, dc); break;
            case 4: by_waves(std::integral_constant<int, 4>{}, dc); break;
            default: by_waves(std::integral_constant<int, 5>{}, dc); break;
        }
    };
    if (d == 64) by_species(std::integral_constant<int, 64>{});
    else by_species(std::integral_constant<int, 128>{});
}
extern "C" int qmll_fchl19_projected_pays(int A, int n, const qmll_fchl_params* prm, int d) {
    return prm && projected_waves(A, n, prm, d) > 0 ? 1 : 0;
}

extern "C" int qmll_prepare_fchl19_project(const float* X, const float* Z, const float* species, const float* model_species, int ne,
                                           const float* cell, const float* inv_cell, const int* atomIDs, const int* molIDs,
                                           const int* natoms, int A, int B, int n, const float* Rs2, const float* Rs3,
                                           const qmll_fchl_params* prm, void* workspace, size_t workspace_bytes, int* types,
                                           int* sort_types, int* sorted_slots, int* type_offsets, float* zero, size_t zero_count,
                                           const float* reductors, int d, float* x, qmll_stream_t stream) {
    FchlArgs a;
    int rc = fill_args(a, X, types, cell, inv_cell, atomIDs, molIDs, natoms, nullptr, nullptr, 0, A, B, n, Rs2, Rs3, prm,
                       "qmll_prepare_fchl19_project");
    if (rc) return rc;
    const long long slots = (long long)B * n;
    const int waves = projected_waves(A, n, prm, d);
    QMLL_REQUIRE(waves > 0, QMLL_ERR_INVALID, "qmll_prepare_fchl19_project: A=%d n=%d d=%d: not a call it takes", A, n, d);
    QMLL_REQUIRE(Z && species && sorted_slots && type_offsets && reductors && x && ne > 0 && (zero || zero_count == 0), QMLL_ERR_INVALID,
                 "qmll_prepare_fchl19_project: null pointer or no elements");
    QMLL_REQUIRE(model_species ? sort_types != nullptr : ne == prm->nspecies, QMLL_ERR_INVALID,
                 "qmll_prepare_fchl19_project: %d elements of %d species without a list of their own", ne, prm->nspecies);
    QMLL_REQUIRE(reinterpret_cast<uintptr_t>(reductors) % 16 == 0, QMLL_ERR_INVALID,
                 "qmll_prepare_fchl19_project: reductors must be 16-byte aligned");
    const int ns = prm->nspecies, np = ns * (ns + 1) / 2, R = ns * prm->nRs2 + 2 * np * prm->nRs3;
    const bool beside = waves == 8 && prepared_beside(A, slots, zero_count, ne, n, prm);
    BatchPrep b = prep_of(Z, species, model_species, ne, A, slots, types, sort_types, sorted_slots, type_offsets, zero, zero_count);
    if (!beside) {
        rc = qmll_prepare_batch(Z, natoms, species, ns, model_species, ne, atomIDs, molIDs, B, n, A, workspace, workspace_bytes, types,
                                sort_types, sorted_slots, type_offsets, zero, zero_count, stream);
        if (rc != QMLL_OK) return rc;
    }
    const long long maxnn = n > 1 ? n - 1 : 1, triples = std::max(maxnn * (maxnn - 1) / 2, 1ll);
    const size_t entries = std::max<size_t>(triples + np * (LEAN_SLOTS - 1), a.cap);
    const size_t lds = std::max(sizeof(float) * (((R + 3) & ~3) + (size_t)waves * d + PREP_ATOMS / 64 + (size_t)8 * a.cap + (3 * entries + 3) / 4 * 4),
                                beside ? sizeof(int) * (size_t)A : 0);                        // (the sort's)
    QMLL_REQUIRE(lds <= LDS_LIMIT, QMLL_ERR_INVALID, "qmll_prepare_fchl19_project: %zu B of LDS needed exceeds %zu", lds, LDS_LIMIT);
    hipStream_t st = (hipStream_t)stream;
    with_projected_shape(ns, d, waves, [&](auto nsc, auto dc, auto wc) {
        constexpr int NS = decltype(nsc)::value, D = decltype(dc)::value, W = decltype(wc)::value;
        if constexpr (W == 8) {
            if (beside) {
                hipLaunchKernelGGL((fchl19_forward_projected_kernel<NS, D, W, true>), dim3(b.groups + A), dim3(64 * W), lds, st, a, b, reductors, x);
                return;
            }
        }
        hipLaunchKernelGGL((fchl19_forward_projected_kernel<NS, D, W, false>), dim3(A), dim3(64 * W), lds, st, a, b, reductors, x);
    });
    QMLL_CHECK_LAUNCH("qmll_prepare_fchl19_project");
    return QMLL_OK;
}

extern "C" int qmll_fchl19_vjp(const float* X, const int* types, const float* cell, const float* inv_cell,
                               const int* atomIDs, const int* molIDs, const int* natoms, const int* nlist,
                               const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2, const float* Rs3,
                               const qmll_fchl_params* prm, const float* grad_rep, float* grad_X,
                               qmll_stream_t stream) {
    return qmll_fchl19_vjp_scaled(X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2,
                                  Rs3, prm, grad_rep, 1.0f, grad_X, stream);
}

extern "C" int qmll_fchl19_vjp_scaled(const float* X, const int* types, const float* cell, const float* inv_cell,
                                      const int* atomIDs, const int* molIDs, const int* natoms, const int* nlist,
                                      const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2,
                                      const float* Rs3, const qmll_fchl_params* prm, const float* grad_rep, float scale,
                                      float* grad_X, qmll_stream_t stream) {
    FchlArgs a;
    int rc = fill_args(a, X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2, Rs3,
                       prm, "qmll_fchl19_vjp");
    if (rc) return rc;
    a.gscale = scale;
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(grad_rep && grad_X, QMLL_ERR_INVALID, "qmll_fchl19_vjp: null gradient pointer");
    const int R = prm->nspecies * prm->nRs2 + prm->nspecies * (prm->nspecies + 1) * prm->nRs3;
    // records of the force copies: the largest number any neighbour count up to cap needs
    a.tcap = 1;
    for (int k = 1; k <= a.cap; ++k) a.tcap = a.tcap < k * force_copies(k) ? k * force_copies(k) : a.tcap;
    const long long maxnn = nlist ? a.cap : a.cap - 1;
    for (int nw = wavefronts_backward(A, maxnn * (maxnn - 1) / 2, a.cap > 54, lean_grids(prm, nlist, n));; nw /= 2) {
        // two records [cap][4], atom indices, force copies, type offsets, grids, the bins' constant factors, the gradient row
        const bool lean4 = nw == 4 && usual_bins(prm);
        const size_t shared = (size_t)9 * a.cap + prm->nspecies + 1 + prm->nRs2 + 2 * prm->nRs3 + R +
                              (lean4 ? (size_t)prm->nspecies * (prm->nspecies + 1) * (LEAN_RS3 - prm->nRs3) : 0);
        const size_t lds = sizeof(float) * (shared + 4 * (size_t)nw * a.tcap + (nw > 1 ? (size_t)prm->nspecies * nw : 0));
        if (lds > LDS_LIMIT && nw > 1) continue;
        hipStream_t st = (hipStream_t)stream;
        if (lds > LDS_LIMIT) {        // beyond about 900 neighbours: one three-float record for each
            a.tcap = a.cap;
            const size_t compact = sizeof(float) * (shared + 3 * (size_t)a.cap);
            QMLL_REQUIRE(compact <= LDS_LIMIT, QMLL_ERR_INVALID,
                         "qmll_fchl19_vjp: %zu B of LDS needed (max_atoms=%d, repsize=%d) exceeds %zu", compact, n, R, LDS_LIMIT);
            hipLaunchKernelGGL((fchl19_vjp_kernel<1, true>), dim3(A), dim3(64), compact, st, a, grad_rep, grad_X);
            break;
        }
        if (nw == 1 && lean_grids(prm, nlist, n)) {
            const int ns = prm->nspecies;
            const size_t lean = sizeof(float) * ((size_t)9 * a.cap + 4 * (size_t)a.tcap + ns * (ns + 1) * LEAN_RS3 + 32 * (ns + 1));
            auto launch = [&](auto nsc) {
                hipLaunchKernelGGL(fchl19_vjp_lean_kernel<decltype(nsc)::value>, dim3(A), dim3(64), lean, st, a, grad_rep, grad_X);
            };
            switch (ns) {
                case 1: launch(std::integral_constant<int, 1>{}); break;
                case 2: launch(std::integral_constant<int, 2>{}); break;
                case 3: launch(std::integral_constant<int, 3>{}); break;
                case 4: launch(std::integral_constant<int, 4>{}); break;
                default: launch(std::integral_constant<int, 5>{}); break;
            }
            break;
        }
        if (lean4) hipLaunchKernelGGL((fchl19_vjp_kernel<4, false, true>), dim3(A), dim3(256), lds, st, a, grad_rep, grad_X);
        else if (nw == 4) hipLaunchKernelGGL(fchl19_vjp_kernel<4>, dim3(A), dim3(256), lds, st, a, grad_rep, grad_X);
        else if (nw == 2) hipLaunchKernelGGL(fchl19_vjp_kernel<2>, dim3(A), dim3(128), lds, st, a, grad_rep, grad_X);
        else hipLaunchKernelGGL(fchl19_vjp_kernel<1>, dim3(A), dim3(64), lds, st, a, grad_rep, grad_X);
        break;
    }
    QMLL_CHECK_LAUNCH("qmll_fchl19_vjp");
    return QMLL_OK;
}

extern "C" int qmll_fchl19_projected_vjp(const float* X, const int* types, const float* cell, const float* inv_cell, const int* atomIDs,
                                         const int* molIDs, const int* natoms, int A, int B, int n, const float* Rs2, const float* Rs3,
                                         const qmll_fchl_params* prm, const float* gx, int nparts, const int* sorted_slots,
                                         const int* type_offsets, const float* reductors, int ne, int d, float scale, float* grad_X,
                                         const float* e_slots, float* energies, qmll_stream_t stream) {
    FchlArgs a;
    int rc = fill_args(a, X, types, cell, inv_cell, atomIDs, molIDs, natoms, nullptr, nullptr, 0, A, B, n, Rs2, Rs3, prm,
                       "qmll_fchl19_projected_vjp");
    if (rc) return rc;
    const int waves = projected_waves(A, n, prm, d);
    QMLL_REQUIRE(waves > 0, QMLL_ERR_INVALID, "qmll_fchl19_projected_vjp: A=%d n=%d d=%d: not a call it takes", A, n, d);
    QMLL_REQUIRE(gx && sorted_slots && type_offsets && reductors && grad_X && ne > 0 && nparts > 0, QMLL_ERR_INVALID,
                 "qmll_fchl19_projected_vjp: null pointer, or no elements or parts");
    QMLL_REQUIRE(reinterpret_cast<uintptr_t>(reductors) % 16 == 0, QMLL_ERR_INVALID,
                 "qmll_fchl19_projected_vjp: reductors must be 16-byte aligned");
    QMLL_REQUIRE(!energies || e_slots, QMLL_ERR_INVALID, "qmll_fchl19_projected_vjp: energies without e_slots");
    a.gscale = scale;
    a.tcap = 1;
    for (int k = 1; k <= a.cap; ++k) a.tcap = std::max(a.tcap, k * force_copies(k));
    const int ns = prm->nspecies, R = ns * prm->nRs2 + ns * (ns + 1) * prm->nRs3;
    const size_t lds = sizeof(float) * (d + ((R + 3) & ~3) + (size_t)9 * a.cap + 4 * waves * (size_t)a.tcap + ns * (ns + 1) * LEAN_RS3 +
                                        32 * (ns + 1) + 3 * waves);
    QMLL_REQUIRE(lds <= LDS_LIMIT, QMLL_ERR_INVALID, "qmll_fchl19_projected_vjp: %zu B of LDS needed exceeds %zu", lds, LDS_LIMIT);
    const ProjectedGradient pg = {gx, nparts, sorted_slots, type_offsets, reductors, ne, A, e_slots, energies};
    const dim3 grid(A + (energies ? (B + waves - 1) / waves : 0));
    with_projected_shape(ns, d, waves, [&](auto nsc, auto dc, auto wc) {
        constexpr int NS = decltype(nsc)::value, D = decltype(dc)::value, W = decltype(wc)::value;
        hipLaunchKernelGGL((fchl19_projected_vjp_kernel<NS, D, W>), grid, dim3(64 * W), lds, (hipStream_t)stream, a, pg, grad_X);
    });
    QMLL_CHECK_LAUNCH("qmll_fchl19_projected_vjp");
    return QMLL_OK;
}

static int jacobian(const float* X, const int* types, const float* cell, const float* inv_cell, const int* atomIDs, const int* molIDs,
                    const int* natoms, const int* nlist, const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2,
                    const float* Rs3, const qmll_fchl_params* prm, float* rep, float* jac, int all_rows, qmll_stream_t stream) {
    FchlArgs a;
    int rc = fill_args(a, X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2, Rs3,
                       prm, "qmll_fchl19_jacobian");
    if (rc) return rc;
    if (A == 0) return QMLL_OK;
    QMLL_REQUIRE(jac != nullptr, QMLL_ERR_INVALID, "qmll_fchl19_jacobian: null output");
    const int R = prm->nspecies * prm->nRs2 + prm->nspecies * (prm->nspecies + 1) * prm->nRs3;
    size_t lds = sizeof(float) * ((size_t)STAGE_ARRAYS * a.cap + prm->nspecies + 1 + 2 * prm->nRs2 + prm->nRs3 + 4 * (size_t)R);
    QMLL_REQUIRE(lds <= LDS_LIMIT, QMLL_ERR_INVALID,
                 "qmll_fchl19_jacobian: %zu B of LDS needed (max_atoms=%d, repsize=%d) exceeds %zu", lds, n, R,
                 LDS_LIMIT);
    // per-triple table while it fits: an atom has at most cap neighbours from a given list and at
    // most max_atoms - 1 otherwise
    const size_t maxnn = nlist ? (size_t)a.cap : (size_t)(a.cap > 1 ? a.cap - 1 : 1);
    const size_t table = sizeof(float) * (JT * (maxnn * (maxnn - 1) / 2) + 4);
    const bool with_table = lds + table <= LDS_LIMIT;
    if (with_table) lds += table;
    // Wavefronts per central atom: as many as give a CU the most, since an atom's rows are a chain of LDS round trips that only other
    // wavefronts fill, and the LDS of its table serves them all.  One wavefront / this, the self rows a third of the work: 3200 atoms of
    // 3 to 29, four elements (three wavefronts) 761 / 393 us; 21000 of 21, three elements (four) 1810 / 1089
    const size_t per_wave = sizeof(float) * 3 * (size_t)R, cu = 160 * 1024;
    int nw = 1;
    for (int w = 2; w <= JW_MOST; ++w) {
        const size_t bytes = lds + sizeof(int) + (w - 1) * per_wave;
        if (bytes <= LDS_LIMIT && (cu / bytes) * w > (cu / (lds + (nw - 1) * per_wave)) * nw) nw = w;
    }
    if (nw > 1) lds += sizeof(int) + (nw - 1) * per_wave;
    if (with_table) hipLaunchKernelGGL(fchl19_jacobian_kernel<true>, dim3(A), dim3(64 * nw), lds, (hipStream_t)stream, a, rep, jac, all_rows);
    else hipLaunchKernelGGL(fchl19_jacobian_kernel<false>, dim3(A), dim3(64 * nw), lds, (hipStream_t)stream, a, rep, jac, all_rows);
    QMLL_CHECK_LAUNCH("qmll_fchl19_jacobian");
    return QMLL_OK;
}

extern "C" int qmll_fchl19_jacobian(const float* X, const int* types, const float* cell, const float* inv_cell,
                                    const int* atomIDs, const int* molIDs, const int* natoms, const int* nlist,
                                    const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2,
                                    const float* Rs3, const qmll_fchl_params* prm, float* rep, float* jac,
                                    qmll_stream_t stream) {
    return jacobian(X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2, Rs3, prm, rep, jac, 0, stream);
}

extern "C" int qmll_fchl19_jacobian_all_rows(const float* X, const int* types, const float* cell, const float* inv_cell,
                                             const int* atomIDs, const int* molIDs, const int* natoms, const int* nlist,
                                             const int* nneigh, int nn_stride, int A, int B, int n, const float* Rs2,
                                             const float* Rs3, const qmll_fchl_params* prm, float* rep, float* jac,
                                             qmll_stream_t stream) {
    return jacobian(X, types, cell, inv_cell, atomIDs, molIDs, natoms, nlist, nneigh, nn_stride, A, B, n, Rs2, Rs3, prm, rep, jac, 1, stream);
}
