// nuosc_pair.hip -- CDNA4 (gfx950) kernels that advance two RK4 stages in one
// pass over the state (2 flavours, the default discretisation).
//
// Open z: the ghost sites of the stencil input are filled by k_pair_ghosts, and
// those of the inner input, which never leaves the chip, by the rule itself (in
// the first step of a segment at the lower end and the last two at the upper).
//
// The stage-by-stage form (k_stage, nuosc_kernels.hip) writes and re-reads
// every stage input: 12 passes over the state per step.  k_pair does stages
// 1+2 and stages 3+4 as two kernels that keep the inner stage input in
// registers and LDS:
//   pair 1: read u       -> Y2 (on chip) -> Y3 = u + dt/2 k2, A = Y2 + u + dt k2
//   pair 2: read Y3, u, A -> Y4 (on chip) -> u' = (A + Y4)/3 + dt/6 k4
// 3 + 4 = 7 passes instead of 12.  In FP64, which is bound by the passes, A is
// not kept either: A = Y2 + 2 Y3 - u and Y2 = u + dt/2 k1, so pair 2 forms k1
// again from the u it reads anyway:
//   pair 1: read u     -> Y2 (on chip) -> Y3
//   pair 2: read Y3, u -> Y4 (on chip) -> u' = (2 Y3 + Y4)/3 + dt/6 (k1 + k4)
// 2 + 3 = 5 passes (320 B per update instead of 768; 512 x 512 x 642: 28.9 ms
// a step stage by stage, 19.3 in 7 passes, 17.8 in 5).  Pair 1 takes 6.7 ms (25
// GB moved, 3.8 TB/s), pair 2 10.7 (38-40 GB); with every load from one z and
// nothing stored they take 5.7 and 9.1, so pair 2 is bound by issuing its
// instructions at 2 waves per SIMD and memory adds a part.  FP32 takes 4.8 and
// 5.1 ms, 3.9 each without memory traffic: a third k in pair 2 would cost more
// than the 2 passes, so there A is kept.  An SSP-RK3 step is a pair and a single stage, 2 + 3 = 5 passes instead of 8:
//   pair 3: read u       -> u1 = u + dt k (on chip) -> u2 = 3/4 u + 1/4 (u1 + dt k)
//   k_lone: read u2, u   -> u' = 1/3 u + 2/3 (u2 + dt k)
//
// What made the passes separate is the interaction term of the inner input Y:
// it needs the velocity moments of Y at each site, a sum over all directions,
// while a block holds 64 of them.  But Y = u + c k(y), and the moments of
// k(y) follow from sums over directions of y itself: the stencil terms are
// linear, and the interaction term is a product of the moments of y with the
// fields, so with the nine sums over w u_a u_b (u = (1, vx, vy, vz);
// vy^2 = 1 - vx^2 - vz^2) of emr, emi and ee - mm, and of their antineutrino
// partners, the moments of k(y) -- and so of Y -- are known at every site
// before any Y is formed:
//   k_pair_totals   adds a site's partial sums over its direction chunks;
//   k_pair_predict  forms from them the moments of y and of Y (per site: the
//                   same stencils on 24 numbers instead of on 8 nv);
//   k_pair          writes the 2 x 27 partial sums of its output.
// The sums are FP64 in both precisions.
//
// The neutrino and antineutrino fields couple only through the moments, so
// the work unit of a wavefront is 4 fields (one of the two) of one x row and
// 64 directions.
#include <hip/hip_runtime.h>

#include "nuosc_dev.h"
#include "nuosc_lanes.h"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace nuosc {
namespace {

constexpr int kF = 4;           // fields of a unit: ee, mm, emr, emi (or the antineutrino ones)
constexpr double kThirdRest = 0x1.5555555555555p-56;   // 1/3 minus its double
constexpr int kMono = 9;        // 1, x, y, z, xx, xy, xz, yz, zz
constexpr int kRec = 3 * kMono; // sums of one unit: [mono][emr, emi, ee - mm]
static_assert(2 * kRec == kPairRec, "record of a site: neutrinos, then antineutrinos");

typedef __attribute__((ext_vector_type(2))) unsigned int pu32x2;
constexpr int kPairRsrc3 = 0x00020000;   // gfx9 raw-buffer descriptor word 3

// AUX: cache policy bits (2: non-temporal)
template <typename T, int AUX = 0>
__device__ __forceinline__ T pld(__amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so) {
    if constexpr (sizeof(T) == 8)
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, AUX));
    else
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, AUX));
}
template <typename T>
__device__ __forceinline__ void pst(T v, __amdgpu_buffer_rsrc_t r, unsigned vo, unsigned so) {
    if constexpr (sizeof(T) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pu32x2, v), r, vo, so, 2);
    else
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, vo, so, 2);
}
// descriptor of the bytes [base, base + bytes); the empty asm keeps it from
// being held in scalar registers across the z loop
__device__ __forceinline__ __amdgpu_buffer_rsrc_t prs(unsigned long long base, unsigned bytes) {
    asm volatile("" : "+s"(base));
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)bytes, kPairRsrc3);
}

// the compiler divides integers in vector registers and may then keep what is
// derived from the quotient there; this puts a wave-uniform value back
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// ---------------------------------------------------------------------------
// Direction sums on the matrix cores.  V_MFMA_F64_4X4X4 multiplies four pairs
// of 4 x 4 matrices; lane l holds A[i = l % 4][q] and B[q][j = l % 4], where
// q = l / 4 runs over the four blocks and the four columns of A (rows of B)
// of each.  With lane l's A value of step t the weighted monomial 4 m + i of
// direction (l & ~3) + t and its B value the field combination j of that
// direction, four steps sum a chunk's 64 directions in four blocks, which two
// DPP adds join.  The combinations move from "lane = direction" to the B
// layout through a small LDS array (each lane needs combination l % 4 of the
// four directions of its quad).  27 sums cost 12 matrix instructions and
// about 45 others; as wavefront reductions they took 160.
// ---------------------------------------------------------------------------
constexpr int kStageStride = 66;   // doubles between the combinations: 16-byte aligned quads, other banks
struct SumStage {
    double v[3 * kStageStride];
};
struct SumTable {
    double2 v[6][64];   // [pair of steps and tiles][lane]: A values 2k, 2k+1 of the 12 = 3 tiles x 4 steps
};

// w mono_n of direction d (0 past nv)
__device__ __forceinline__ double weighted_mono(const Geometry& g, int d, int n) {
    if (d >= g.nv || n >= kMono) return 0.0;
    const double x = g.vx[d], y = g.vy[d], z = g.vz[d], w = g.vw[d];
    const double p = n == 0 || n == 1 || n == 2 || n == 3 ? 1.0 : (n < 7 ? x : (n == 7 ? y : z));
    const double q = n == 0 ? 1.0 : (n == 1 || n == 4 ? x : (n == 2 || n == 5 ? y : z));
    return p * q * w;
}
// the table entries of one lane, chunk ch
__device__ __forceinline__ void fill_table(const Geometry& g, SumTable& t, int ch, int lane) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        double e[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int m = (2 * k + h) / 4, s = (2 * k + h) % 4;
            e[h] = weighted_mono(g, ch * 64 + (lane & ~3) + s, 4 * m + (lane & 3));
        }
        t.v[k][lane] = make_double2(e[0], e[1]);
    }
}

__device__ __forceinline__ double dpp_add_ror(double x, bool eight) {
    // x + x of lane +-8 / +-4 within the 16-lane row
    return eight ? x + dpp_f64<kDppRowRor8, 0xF>(x, x) : x + dpp_f64<kDppRowRor4, 0xF>(x, x);
}

// Direction sums of (c0, c1, c2) over the chunk, stored as one record of 27
// doubles at so under descriptor rp (vrec: the lane's offset from sum_offset).
__device__ __forceinline__ void direction_sums(double c0, double c1, double c2, SumStage& st, const SumTable& tab,
                                               int lane, __amdgpu_buffer_rsrc_t rp, unsigned vrec, unsigned so) {
    st.v[lane] = c0;
    st.v[kStageStride + lane] = c1;
    st.v[2 * kStageStride + lane] = c2;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    // (lanes of the unused fourth column read the third combination)
    const double* q = &st.v[min(lane & 3, 2) * kStageStride + (lane & ~3)];
    const double b[4] = {q[0], q[1], q[2], q[3]};
    double d[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
        const double2 a01 = tab.v[2 * m][lane], a23 = tab.v[2 * m + 1][lane];
        double acc = __builtin_amdgcn_mfma_f64_4x4x4f64(a01.x, b[0], 0.0, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(a01.y, b[1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f64_4x4x4f64(a23.x, b[2], acc, 0, 0, 0);
        d[m] = __builtin_amdgcn_mfma_f64_4x4x4f64(a23.y, b[3], acc, 0, 0, 0);
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) d[m] = dpp_add_ror(dpp_add_ror(d[m], true), false);
    // every block's lanes hold the joined sums: block m stores tile m
    const int blk = (lane >> 2) & 3;
    const double v = blk == 0 ? d[0] : (blk == 1 ? d[1] : d[2]);
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(pu32x2, v), rp, vrec, so, 0);
}
// lane l of D holds row i = l / 16, column j = l % 4 of block (l / 4) % 4:
// sum 4 m + i of combination j; lanes without one point past the record array
__device__ __forceinline__ unsigned sum_offset(int lane, unsigned past) {
    const int m = (lane >> 2) & 3, i = lane >> 4, j = lane & 3, n = 4 * m + i;
    return (m < 3 && j < 3 && n < kMono) ? (unsigned)(n * 3 + j) * 8u : past;
}

// ---------------------------------------------------------------------------
// the stage pair
// ---------------------------------------------------------------------------
template <typename T>
struct PairArgs {
    Geometry g;
    unsigned long long y;      // stencil input (stored x row 0): u (pairs 1, 3), Y3 (pair 2), u2 (lone stage)
    unsigned long long u;      // pair 2, lone stage: u
    unsigned long long a;      // A (FP32): written by pair 1, read by pair 2
    unsigned long long out;    // Y3 (pair 1), u2 (pair 3), u' (pair 2, lone stage); no input of the pass
    unsigned long long m1, m2; // moment records of y and of the inner input: [site][kMomStride]
    unsigned long long m0;     // pair 2: of u
    unsigned long long part;   // partial sums of out: [site][chunk][2][kRec]
    unsigned long long gin;    // open z: inflow values of the inner input's ghost sites, [end][depth][8][nvp]
    double c1, c2, cA;         // inner input u + c1 k; output's and A's factors of k (pair 3, lone stage:
                               // output c2 u + cA (y + c1 k))
    int zlen, xgroups, nunits;
};

// FP64: pair 2 forms k1 again instead of reading A
template <typename T, int PAIR>
constexpr bool kAgain = sizeof(T) == 8 && PAIR == 2;

// x rows a block writes: R, from R + 4 rows of the inner input (a wavefront
// each) and R + 8 of y; and the waves per SIMD its registers allow.  FP64: 12
// waves (3 per SIMD, 168 VGPRs) with a slab of 137 KB; pair 2 holds a z window
// of u as well (230 VGPRs, so 8 waves, 2 per SIMD; 131 KB).  FP32: 16 waves (4 per SIMD): fewer
// edge rows for the row (12 waves at 5 per SIMD took 14.6 instead of 11.5 ms
// per step at 512 x 512 x 642).
template <typename T, int PAIR>
struct PairShape {
    static constexpr int R = sizeof(T) == 4 ? 12 : (kAgain<T, PAIR> ? 4 : 8);
    static constexpr int SimdWaves = sizeof(T) == 4 ? 4 : (kAgain<T, PAIR> ? 2 : 3);
};

template <typename T, int R, bool AGAIN>
struct PairSlab {
    T y[2][R + 9][kF][64];   // rows -4 .. R+3 of y at the inner input's z, and a slot idle lanes write
    T m[2][R + 4][kF][64];   // rows -2 .. R+1 of the inner input
    T u[AGAIN ? 2 : 0][R + 4][kF][64];   // the same rows of u
    SumTable tab;
    SumStage st[R];
};
// one x row: no neighbours to share
template <int W>
struct PairRowLds {
    SumTable tab[W];
    SumStage st[W];
};

// Per-direction and physics factors of k(y)
template <typename T>
struct PairConst {
    double nvx, nvy, nvz;   // minus the direction
    T fx, fz;          // -v / (12 h)
    T kx, kz, k6;      // -ko / (16 h) per axis; 6 (kx + kz)
};

template <typename T>
__device__ __forceinline__ PairConst<T> pair_const(const Geometry& g, int pv) {
    PairConst<T> k;
    k.nvx = -g.vx[pv];
    k.nvy = -g.vy[pv];
    k.nvz = -g.vz[pv];
    k.fx = (T)(k.nvx / g.twelve_dx);
    k.fz = (T)(k.nvz / g.twelve_dz);
    k.kx = (T)g.ko_x;
    k.kz = (T)g.ko_z;
    k.k6 = (T)(6 * (g.ko_x + g.ko_z));
    return k;
}

// Interaction and vacuum terms as one precession: with the projections A, B, C
// of the site's moments (INP, nuosc_class.cpp:187),
//   k_ee = 2 (q emi + b emr), k_mm = -k_ee, k_emr = -(b d + c emi),
//   k_emi = c emr - q d,  d = ee - mm,
//   q = mu A - pmo st, b = mu B, c = mu C + 2 pmo ct
// (the records of the pair kernels hold mu times the moments, with the vacuum
// terms added to the first of A and of C: k_pair_predict)
// (the terms of nuosc_class.cpp:193-200, 280-287 collected).
template <typename T>
struct Precession {
    T q, b, c;
};
// x: the site's record, value n in lane n of every 16-lane row.  The products
// take it by DPP row_newbcast (64-bit operations have that control), four
// instructions a projection; the compiler forms a broadcast as two moves
// instead (24 per stage), and records in scalar registers (three moves) cost a
// scalar load that no register is free to prefetch.  (The s_nop covers a DPP
// read of x behind the instruction that wrote it.)
#define NUOSC_BC(n) " row_newbcast:" #n " row_mask:0xf bank_mask:0xf\n\t"
template <typename T>
__device__ __forceinline__ Precession<T> precession(const PairConst<T>& k, double x) {
    double A, B, C;
    asm("s_nop 1\n\t"
        "v_mov_b64_dpp %0, %3" NUOSC_BC(0)
        "v_mov_b64_dpp %1, %3" NUOSC_BC(4)
        "v_mov_b64_dpp %2, %3" NUOSC_BC(8)
        "v_fmac_f64_dpp %0, %3, %4" NUOSC_BC(1)
        "v_fmac_f64_dpp %1, %3, %4" NUOSC_BC(5)
        "v_fmac_f64_dpp %2, %3, %4" NUOSC_BC(9)
        "v_fmac_f64_dpp %0, %3, %5" NUOSC_BC(2)
        "v_fmac_f64_dpp %1, %3, %5" NUOSC_BC(6)
        "v_fmac_f64_dpp %2, %3, %5" NUOSC_BC(10)
        "v_fmac_f64_dpp %0, %3, %6" NUOSC_BC(3)
        "v_fmac_f64_dpp %1, %3, %6" NUOSC_BC(7)
        "v_fmac_f64_dpp %2, %3, %6" NUOSC_BC(11)
        : "=&v"(A), "=&v"(B), "=&v"(C)
        : "v"(x), "v"(k.nvx), "v"(k.nvy), "v"(k.nvz));
    return Precession<T>{(T)A, (T)B, (T)C};
}
#undef NUOSC_BC

// k(y) of the 4 fields: c centre values, z neighbours, x neighbours through
// the callable.  The stencils (nuosc_class.cpp:122-123, 182-183) are taken on
// differences and sums of opposite neighbours, so that the advection term
// keeps the exact differences, and added to the local terms one by one.
template <typename T, typename XN>
__device__ __forceinline__ void rhs_unit(const PairConst<T>& k, const Precession<T>& r, const T (&c)[kF],
                                         const T (&zm2)[kF], const T (&zm1)[kF], const T (&zp1)[kF],
                                         const T (&zp2)[kF], XN xn, T (&out)[kF]) {
    const T d = c[0] - c[1], ee = (T)2 * (r.q * c[3] + r.b * c[2]);
    const T loc[kF] = {ee, -ee, -(r.b * d + r.c * c[3]), r.c * c[2] - r.q * d};
#pragma unroll
    for (int f = 0; f < kF; ++f) {
        T xm2, xm1, xp1, xp2;
        xn(f, xm2, xm1, xp1, xp2);
        T t = loc[f] + k.k6 * c[f];
        t += k.kz * ((zm2[f] + zp2[f]) - (T)4 * (zm1[f] + zp1[f]));
        t += k.kx * ((xm2 + xp2) - (T)4 * (xm1 + xp1));
        t += k.fz * ((zm2[f] - zp2[f]) - (T)8 * (zm1[f] - zp1[f]));
        t += k.fx * ((xm2 - xp2) - (T)8 * (xm1 - xp1));
        out[f] = t;
    }
}

// Open z: inflow values of the inner input at the ghost site of this depth past
// one end; those past the upper end are kept in LDS (glds): a load in the z
// loop that only its last steps need would have to be waited for in each.
template <typename T>
__device__ __forceinline__ void inflow_values(const PairArgs<T>& a, int ch, int grp, int end, int depth, T (&v)[kF]) {
    const int pv = min(ch * 64 + (int)(threadIdx.x & 63), a.g.nv - 1);
    const T* p = (const T*)a.gin + (long long)((end * 2 + depth - 1) * kNVar + grp * kF) * a.g.nvp + pv;
#pragma unroll
    for (int f = 0; f < kF; ++f) v[f] = p[(long long)f * a.g.nvp];
}
template <typename T, bool OPEN, int W>
struct GhostLds {
    T v[W][2][kF][64];
    __device__ __forceinline__ const T (*get(int w) const)[kF][64] { return v[w]; }
    __device__ __forceinline__ void fill(const PairArgs<T>& a, int ch, int grp, int w) {
        T x[kF];
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            inflow_values(a, ch, grp, 1, d + 1, x);
#pragma unroll
            for (int f = 0; f < kF; ++f) v[w][d][f][threadIdx.x & 63] = x[f];
        }
    }
};
template <typename T, int W>
struct GhostLds<T, false, W> {
    __device__ __forceinline__ const T (*get(int) const)[kF][64] { return nullptr; }
    __device__ __forceinline__ void fill(const PairArgs<T>&, int, int, int) {}
};

// One wavefront of a pair: x row `row`, unit (chunk ch, neutrinos grp = 0 or
// antineutrinos 1), z segment [j0, j1).  Step j forms the inner input at
// z = j + 2 and, from step j0 on, the output at z = j; the four steps before
// j0 fill the inner input's z window.
//   OUT   the wave writes its row; otherwise the row only feeds neighbours
//         (and the wave loads an edge row of y)
//   NOX   one x row: x neighbours are the point itself, no slab, no barrier
//   OPEN  open z (a form of its own: the periodic one has no branch in its steps)
// Per step each wave puts its row of y at z = j + 2 and of the inner input at
// z = j into the slab of the step's parity, passes the one barrier, and reads
// its x neighbours; the other parity's slab is rewritten only after the next
// barrier, which every wave reaches after its reads.  The rows of y and u that
// step j loads are used from step j + 1 on, so a wave does not wait for what
// it has just asked for: the waves of a block move in step, and one block
// fills a CU's registers.  Edge rows are loaded at the z at which the
// neighbouring blocks load them as their own (L2 hits).
// The z windows are rings of six slots and a step is compiled for each of the
// six phases, so that no register is moved to shift a window (54 of 354
// vector instructions per step before).
template <typename T, int PAIR, bool OUT, bool NOX, bool OPEN, typename LDS>
__device__ __forceinline__ void pair_wave(const PairArgs<T>& a, int row, int ch, int grp, int j0, int j1, int slot_m,
                                          int erow, int slot_e, SumTable& tab, SumStage& sst, LDS* lds,
                                          const T (*glds)[kF][64]) {
    const Geometry& g = a.g;
    const int lane = threadIdx.x & 63, nz = g.nz, zo = OPEN ? g.zoff : 0;
    const unsigned rowb = (unsigned)g.nvp * (unsigned)sizeof(T);
    const unsigned siteb = (unsigned)(g.srec * (long long)sizeof(T));
    const unsigned long long xrowb = (unsigned long long)g.xrow * sizeof(T);
    const unsigned gofs = (unsigned)(grp * kF) * rowb;
    const unsigned long long rbase = (unsigned long long)(row + kXg) * xrowb + gofs;
    const unsigned long long ebase = (unsigned long long)(max(erow, 0) + kXg) * xrowb + gofs;
    const unsigned rbytes = (unsigned)xrowb - gofs;
    const int pv = min(ch * 64 + lane, g.nv - 1);   // lanes past nv work on the last direction (and store its bits)
    const unsigned vo = (unsigned)pv * (unsigned)sizeof(T);
    const unsigned ve = erow >= 0 ? vo : rbytes;    // no edge row: past the range, nothing is fetched
    const unsigned zrec = (unsigned)(g.nch * kPairRec * 8);   // bytes of a site's partial records
    const unsigned rec0 = (unsigned)(ch * kPairRec + grp * kRec) * 8;
    const unsigned long long prow = a.part + (unsigned long long)row * nz * zrec + rec0;
    const unsigned pbytes = (unsigned)nz * zrec - rec0;
    const unsigned vrec = sum_offset(lane, pbytes);
    const unsigned long long mrow = (unsigned long long)row * nz * (kMomStride * 8);
    const unsigned mbytes = (unsigned)nz * (kMomStride * 8), vm = (unsigned)(lane & 15) * 8;
    const PairConst<T> k = pair_const<T>(g, pv);
    const T c1 = (T)a.c1, c2 = (T)a.c2, cA = (T)a.cA;

    T U[6][kF];    // y of the own row, z = j .. j+4, and j+5 on its way: slot (phase + z - j) % 6
    T Y[6][kF];    // inner input, z = j-2 .. j+2: slot (phase + 2 + z - j) % 6 (not OUT: from j on)
    T E[6][kF];    // not OUT: edge row of y, z = j+2 .. j+5, in the slots of U
    T uc[kF];      // pair 2 (FP32): u at z = j+2 (of the next step, once used)
    T W[6][kF];    // pair 2 (FP64): u of the own row, z = j-2 .. j+2, and j+3 on its way: the slots of Y
    // step j's site j + q: wrapped, or (open z) within the two ghost sites at
    // each end (those of the first and last steps that lie further out are not used)
    auto at = [&](int jj, int q) { return OPEN ? max(-2, min(jj + q, nz + 1)) : wrapi(jj + q, nz); };
    auto next = [&](int z, int jj, int q) { return OPEN ? at(jj, q) : (z + 1 == nz ? 0 : z + 1); };
    auto load = [&](unsigned long long base, unsigned v, int z, T (&x)[kF]) {
        const __amdgpu_buffer_rsrc_t r = prs(base, rbytes);
#pragma unroll
        for (int f = 0; f < kF; ++f) x[f] = pld<T>(r, v, (unsigned)(z + zo) * siteb + f * rowb);
    };
    int j = j0 - 4;   // the step; z5, z3, z1: wrapped j+5, j+3, j+1
    int z5 = uniform(at(j, 5)), z3 = uniform(at(j, 3)), z1 = uniform(at(j, 1));
    const int z2 = uniform(at(j, 2));
#pragma unroll
    for (int q = 0; q < 5; ++q) load(a.y + rbase, vo, at(j, q), U[q]);
    if constexpr (!OUT && !NOX) {
#pragma unroll
        for (int q = 2; q < 5; ++q) load(a.y + ebase, ve, at(j, q), E[q]);
    }
    constexpr bool AGAIN = kAgain<T, PAIR>;
    // moment records of this step and the next: of y at z = j+2, of the inner
    // input and (FP64 pair 2) of u at z = j
    auto moment = [&](unsigned long long m, int z) {
        if constexpr (OPEN) z = max(0, min(z, nz - 1));   // (no k is wanted at a ghost site)
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(prs(m + mrow, mbytes), vm,
                                                                               (unsigned)z * (kMomStride * 8), 0));
    };
    double M1[2], M2[2] = {0.0, 0.0}, M0[2] = {0.0, 0.0};
    M1[0] = moment(a.m1, z2);
    if constexpr (AGAIN) load(a.u + rbase, vo, z2, W[4]);
    else if constexpr (PAIR == 2) load(a.u + rbase, vo, z2, uc);
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int f = 0; f < kF; ++f) Y[q][f] = (T)0;

    // open z: the inner input at the ghost site of this depth past one end: the
    // inflow value v, or extrapolated from the edge sites e0, e1, e2
    auto ghost = [&](int end, int depth, T v, T e0, T e1, T e2) {
        const bool in = end == 0 ? k.nvz < 0.0 : k.nvz > 0.0;
        return in ? v : (T)open_extrapolate(depth, (double)e0, (double)e1, (double)e2);
    };
    // phase P: the step's number modulo 6; WRITE: step j0 or later; BEGIN: step j0 (open z)
    auto step = [&](auto phase, auto write) {
        constexpr int P = decltype(phase)::value;
        constexpr bool WRITE = decltype(write)::value != 0, BEGIN = decltype(write)::value == 2;
        constexpr int b = P & 1;
        const auto& U0 = U[P % 6];
        const auto& U1 = U[(P + 1) % 6];
        const auto& U2 = U[(P + 2) % 6];
        const auto& U3 = U[(P + 3) % 6];
        const auto& U4 = U[(P + 4) % 6];
        auto& Y0 = Y[P % 6];
        auto& Y1 = Y[(P + 1) % 6];
        const auto& Y2 = Y[(P + 2) % 6];
        const auto& Y3 = Y[(P + 3) % 6];
        auto& Y4 = Y[(P + 4) % 6];
        // ---- loads for the next steps (A: for the end of this one)
        load(a.y + rbase, vo, z5, U[(P + 5) % 6]);
        if constexpr (!OUT && !NOX) load(a.y + ebase, ve, z5, E[(P + 5) % 6]);
        if constexpr (AGAIN) load(a.u + rbase, vo, z3, W[(P + 5) % 6]);
        T ac[kF];
        if constexpr (PAIR == 2 && !AGAIN && WRITE) {
            const __amdgpu_buffer_rsrc_t ra = prs(a.a + rbase, rbytes);
#pragma unroll
            for (int f = 0; f < kF; ++f) ac[f] = pld<T, 2>(ra, vo, (unsigned)(j + zo) * siteb + f * rowb);
        }
        // moment records of the next step
        M1[b ^ 1] = moment(a.m1, z3);
        if constexpr (OUT) M2[b ^ 1] = moment(a.m2, z1);
        if constexpr (OUT && AGAIN) M0[b ^ 1] = moment(a.m0, z1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!NOX) {
#pragma unroll
            for (int f = 0; f < kF; ++f) lds->y[b][slot_m + 2][f][lane] = U2[f];
#pragma unroll
            for (int f = 0; f < kF; ++f) lds->m[b][slot_m][f][lane] = Y2[f];
            if constexpr (AGAIN && WRITE) {
#pragma unroll
                for (int f = 0; f < kF; ++f) lds->u[b][slot_m][f][lane] = W[(P + 2) % 6][f];
            }
            if constexpr (!OUT) {
#pragma unroll
                for (int f = 0; f < kF; ++f) lds->y[b][slot_e][f][lane] = E[(P + 2) % 6][f];
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
        {   // ---- the inner input at z = j + 2
            const Precession<T> r1 = precession(k, M1[b]);
            T kk[kF];
            rhs_unit<T>(k, r1, U2, U0, U1, U3, U4,
                        [&](int f, T& xm2, T& xm1, T& xp1, T& xp2) {
                            if constexpr (NOX) {
                                xm2 = xm1 = xp1 = xp2 = U2[f];
                            } else {
                                xm2 = lds->y[b][slot_m][f][lane];
                                xm1 = lds->y[b][slot_m + 1][f][lane];
                                xp1 = lds->y[b][slot_m + 3][f][lane];
                                xp2 = lds->y[b][slot_m + 4][f][lane];
                            }
                        },
                        kk);
#pragma unroll
            for (int f = 0; f < kF; ++f) {
                Y4[f] = (PAIR != 2 ? U2[f] : (AGAIN ? W[(P + 4) % 6][f] : uc[f])) + c1 * kk[f];
                // (not OUT: computed here, not sunk to its use two steps on,
                // which kept every operand alive and spilled)
                if constexpr (!OUT) asm volatile("" : "+v"(Y4[f]));
            }
        }
        if constexpr (OPEN && OUT) {   // ghost sites past the upper end
            if (j + 2 >= nz) {
                const int past = j + 2 - nz;
#pragma unroll
                for (int f = 0; f < kF; ++f)
                    Y4[f] = ghost(1, past + 1, glds[past][f][lane], past ? Y2[f] : Y3[f], past ? Y1[f] : Y2[f],
                                  past ? Y0[f] : Y1[f]);
            }
        }
        if constexpr (PAIR == 2 && !AGAIN) {
            load(a.u + rbase, vo, z3, uc);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (OPEN && OUT && BEGIN) {   // and below the lower one
            if (j < 2) {
                T gv1[kF], gv2[kF];
                inflow_values(a, ch, grp, 0, 1, gv1);
                inflow_values(a, ch, grp, 0, 2, gv2);
#pragma unroll
                for (int f = 0; f < kF; ++f) {
                    const T y1 = j == 0 ? ghost(0, 1, gv1[f], Y2[f], Y3[f], Y4[f]) : Y1[f];
                    Y0[f] = j == 0 ? ghost(0, 2, gv2[f], Y2[f], Y3[f], Y4[f]) : ghost(0, 1, gv1[f], Y1[f], Y2[f], Y3[f]);
                    Y1[f] = y1;
                }
            }
        }
        if constexpr (OUT && WRITE) {   // ---- the output at z = j
            const Precession<T> r2 = precession(k, M2[b]);
            T kk[kF], yo[kF];
            rhs_unit<T>(k, r2, Y2, Y0, Y1, Y3, Y4,
                        [&](int f, T& xm2, T& xm1, T& xp1, T& xp2) {
                            if constexpr (NOX) {
                                xm2 = xm1 = xp1 = xp2 = Y2[f];
                            } else {
                                xm2 = lds->m[b][slot_m - 2][f][lane];
                                xm1 = lds->m[b][slot_m - 1][f][lane];
                                xp1 = lds->m[b][slot_m + 1][f][lane];
                                xp2 = lds->m[b][slot_m + 2][f][lane];
                            }
                        },
                        kk);
            const unsigned so = (unsigned)(j + zo) * siteb;
            const __amdgpu_buffer_rsrc_t ro = prs(a.out + rbase, rbytes);
            // (1/3 in two parts: a third rounded to T alone grows u by 3e-8 (FP32)
            // or 6e-17 of itself every step)
            const T third = (T)(1.0 / 3.0), rest = sizeof(T) == 4 ? (T)(1.0 / 3.0 - (double)third) : (T)kThirdRest;
            if constexpr (PAIR == 1) {   // Y3 = u + dt/2 k2, A = Y2 + u + dt k2
                const __amdgpu_buffer_rsrc_t ra = prs(a.a + rbase, rbytes);
#pragma unroll
                for (int f = 0; f < kF; ++f) {
                    yo[f] = U0[f] + c2 * kk[f];
                    if constexpr (!kAgain<T, 2>) pst<T>((Y2[f] + U0[f]) + cA * kk[f], ra, vo, so + f * rowb);
                }
            } else if constexpr (AGAIN) {   // u' = (2 Y3 + Y4) / 3 + dt/6 (k1 + k4)
                const Precession<T> r0 = precession(k, M0[b]);
                const auto& W2 = W[(P + 2) % 6];
                T k1[kF];
                rhs_unit<T>(k, r0, W2, W[P % 6], W[(P + 1) % 6], W[(P + 3) % 6], W[(P + 4) % 6],
                            [&](int f, T& xm2, T& xm1, T& xp1, T& xp2) {
                                if constexpr (NOX) {
                                    xm2 = xm1 = xp1 = xp2 = W2[f];
                                } else {
                                    xm2 = lds->u[b][slot_m - 2][f][lane];
                                    xm1 = lds->u[b][slot_m - 1][f][lane];
                                    xp1 = lds->u[b][slot_m + 1][f][lane];
                                    xp2 = lds->u[b][slot_m + 2][f][lane];
                                }
                            },
                            k1);
#pragma unroll
                for (int f = 0; f < kF; ++f) {
                    const T s = (T)2 * U0[f] + Y2[f];
                    yo[f] = s * third + (s * rest + c2 * (k1[f] + kk[f]));
                }
            } else if constexpr (PAIR == 3) {   // u2 = 3/4 u + 1/4 (u1 + dt k)
#pragma unroll
                for (int f = 0; f < kF; ++f) yo[f] = c2 * U0[f] + cA * (Y2[f] + c1 * kk[f]);
            } else {                     // u' = (A + Y4) / 3 + dt/6 k4
#pragma unroll
                for (int f = 0; f < kF; ++f) {
                    const T s = ac[f] + Y2[f];
                    yo[f] = s * third + (s * rest + c2 * kk[f]);
                }
            }
#pragma unroll
            for (int f = 0; f < kF; ++f) pst<T>(yo[f], ro, vo, so + f * rowb);
            direction_sums((double)yo[2], (double)yo[3], (double)yo[0] - (double)yo[1], sst, tab, lane,
                           prs(prow, pbytes), vrec, (unsigned)j * zrec);
        }
        ++j;
        z5 = next(z5, j, 5);
        z3 = next(z3, j, 3);
        z1 = next(z1, j, 1);
    };
    using std::integral_constant;
    step(integral_constant<int, 0>{}, integral_constant<int, 0>{});
    step(integral_constant<int, 1>{}, integral_constant<int, 0>{});
    step(integral_constant<int, 2>{}, integral_constant<int, 0>{});
    step(integral_constant<int, 3>{}, integral_constant<int, 0>{});
    if constexpr (OPEN) {   // (step j0 by itself: only there can the lower end lie in the window)
        step(integral_constant<int, 4>{}, integral_constant<int, 2>{});
        while (j != j1) {
            step(integral_constant<int, 5>{}, integral_constant<int, 1>{});
            if (j == j1) break;
            step(integral_constant<int, 0>{}, integral_constant<int, 1>{});
            if (j == j1) break;
            step(integral_constant<int, 1>{}, integral_constant<int, 1>{});
            if (j == j1) break;
            step(integral_constant<int, 2>{}, integral_constant<int, 1>{});
            if (j == j1) break;
            step(integral_constant<int, 3>{}, integral_constant<int, 1>{});
            if (j == j1) break;
            step(integral_constant<int, 4>{}, integral_constant<int, 1>{});
        }
        return;
    }
    for (;;) {
        step(integral_constant<int, 4>{}, integral_constant<int, 1>{});
        if (j == j1) break;
        step(integral_constant<int, 5>{}, integral_constant<int, 1>{});
        if (j == j1) break;
        step(integral_constant<int, 0>{}, integral_constant<int, 1>{});
        if (j == j1) break;
        step(integral_constant<int, 1>{}, integral_constant<int, 1>{});
        if (j == j1) break;
        step(integral_constant<int, 2>{}, integral_constant<int, 1>{});
        if (j == j1) break;
        step(integral_constant<int, 3>{}, integral_constant<int, 1>{});
        if (j == j1) break;
    }
}

// A wavefront of a lone stage (SSP-RK3's last): the output at z = j from y at
// z = j-2 .. j+2 and u at z = j, with the loads, the slab of y rows and the ring
// of phases of pair_wave.  All R + 4 rows of a block are output rows (put:
// inside the grid); its first and last two waves also load the rows beyond.
template <typename T, bool NOX, bool OPEN, typename LDS>
__device__ __forceinline__ void lone_wave(const PairArgs<T>& a, int row, bool put, int ch, int grp, int j0, int j1,
                                          int slot, int erow, int slot_e, SumTable& tab, SumStage& sst, LDS* lds) {
    const Geometry& g = a.g;
    const int lane = threadIdx.x & 63, nz = g.nz, zo = OPEN ? g.zoff : 0;
    const unsigned rowb = (unsigned)g.nvp * (unsigned)sizeof(T);
    const unsigned siteb = (unsigned)(g.srec * (long long)sizeof(T));
    const unsigned long long xrowb = (unsigned long long)g.xrow * sizeof(T);
    const unsigned gofs = (unsigned)(grp * kF) * rowb;
    const unsigned long long rbase = (unsigned long long)(row + kXg) * xrowb + gofs;
    const unsigned long long ebase = (unsigned long long)(max(erow, 0) + kXg) * xrowb + gofs;
    const unsigned rbytes = (unsigned)xrowb - gofs;
    const int pv = min(ch * 64 + lane, g.nv - 1);
    const unsigned vo = (unsigned)pv * (unsigned)sizeof(T);
    const unsigned ve = erow >= 0 ? vo : rbytes, vs = put ? vo : rbytes;
    const unsigned zrec = (unsigned)(g.nch * kPairRec * 8);
    const unsigned rec0 = (unsigned)(ch * kPairRec + grp * kRec) * 8;
    const unsigned long long prow = a.part + (unsigned long long)row * nz * zrec + rec0;
    const unsigned pbytes = (unsigned)nz * zrec - rec0;
    const unsigned vrec = put ? sum_offset(lane, pbytes) : pbytes;
    const unsigned long long mrow = (unsigned long long)row * nz * (kMomStride * 8);
    const unsigned mbytes = (unsigned)nz * (kMomStride * 8), vm = (unsigned)(lane & 15) * 8;
    const PairConst<T> k = pair_const<T>(g, pv);
    const T c1 = (T)a.c1, c2 = (T)a.c2, cA = (T)a.cA;

    T U[6][kF];   // y of the own row, z = j-2 .. j+2, and j+3 on its way: slot (phase + 2 + z - j) % 6
    T E[6][kF];   // edge row of y, z = j .. j+3, in the slots of U
    auto at = [&](int jj, int q) { return OPEN ? max(-2, min(jj + q, nz + 1)) : wrapi(jj + q, nz); };   // as pair_wave
    auto next = [&](int z, int jj, int q) { return OPEN ? at(jj, q) : (z + 1 == nz ? 0 : z + 1); };
    auto load = [&](unsigned long long base, unsigned v, int z, T (&x)[kF]) {
        const __amdgpu_buffer_rsrc_t r = prs(base, rbytes);
#pragma unroll
        for (int f = 0; f < kF; ++f) x[f] = pld<T>(r, v, (unsigned)(z + zo) * siteb + f * rowb);
    };
    int j = j0;
    int z3 = uniform(at(j, 3)), z1 = uniform(at(j, 1));
    auto moment = [&](int z) {
        if constexpr (OPEN) z = min(z, nz - 1);
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(prs(a.m1 + mrow, mbytes), vm,
                                                                               (unsigned)z * (kMomStride * 8), 0));
    };
    double M1[2] = {moment(j), 0.0};
#pragma unroll
    for (int q = 0; q < 5; ++q) load(a.y + rbase, vo, uniform(at(j, q - 2)), U[q]);
    if constexpr (!NOX) {
#pragma unroll
        for (int q = 2; q < 5; ++q) load(a.y + ebase, ve, uniform(at(j, q - 2)), E[q]);
    }
    auto step = [&](auto phase) {
        constexpr int P = decltype(phase)::value;
        constexpr int b = P & 1;
        const auto& U2 = U[(P + 2) % 6];
        load(a.y + rbase, vo, z3, U[(P + 5) % 6]);
        if constexpr (!NOX) load(a.y + ebase, ve, z3, E[(P + 5) % 6]);
        T uc[kF];
        {
            const __amdgpu_buffer_rsrc_t ru = prs(a.u + rbase, rbytes);
#pragma unroll
            for (int f = 0; f < kF; ++f) uc[f] = pld<T, 2>(ru, vo, (unsigned)(j + zo) * siteb + f * rowb);
        }
        M1[b ^ 1] = moment(z1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (!NOX) {
#pragma unroll
            for (int f = 0; f < kF; ++f) lds->y[b][slot + 2][f][lane] = U2[f];
#pragma unroll
            for (int f = 0; f < kF; ++f) lds->y[b][slot_e][f][lane] = E[(P + 2) % 6][f];
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        }
        const Precession<T> r1 = precession(k, M1[b]);
        T kk[kF], yo[kF];
        rhs_unit<T>(k, r1, U2, U[P % 6], U[(P + 1) % 6], U[(P + 3) % 6], U[(P + 4) % 6],
                    [&](int f, T& xm2, T& xm1, T& xp1, T& xp2) {
                        if constexpr (NOX) {
                            xm2 = xm1 = xp1 = xp2 = U2[f];
                        } else {
                            xm2 = lds->y[b][slot][f][lane];
                            xm1 = lds->y[b][slot + 1][f][lane];
                            xp1 = lds->y[b][slot + 3][f][lane];
                            xp2 = lds->y[b][slot + 4][f][lane];
                        }
                    },
                    kk);
        const __amdgpu_buffer_rsrc_t ro = prs(a.out + rbase, rbytes);
#pragma unroll
        for (int f = 0; f < kF; ++f) {
            yo[f] = c2 * uc[f] + cA * (U2[f] + c1 * kk[f]);
            pst<T>(yo[f], ro, vs, (unsigned)(j + zo) * siteb + f * rowb);
        }
        direction_sums((double)yo[2], (double)yo[3], (double)yo[0] - (double)yo[1], sst, tab, lane, prs(prow, pbytes),
                       vrec, (unsigned)j * zrec);
        ++j;
        z3 = next(z3, j, 3);
        z1 = next(z1, j, 1);
    };
    using std::integral_constant;
    for (;;) {
        step(integral_constant<int, 0>{});
        if (j == j1) break;
        step(integral_constant<int, 1>{});
        if (j == j1) break;
        step(integral_constant<int, 2>{});
        if (j == j1) break;
        step(integral_constant<int, 3>{});
        if (j == j1) break;
        step(integral_constant<int, 4>{});
        if (j == j1) break;
        step(integral_constant<int, 5>{});
        if (j == j1) break;
    }
}

// logical block -> (neutrinos or antineutrinos fastest, x group, chunk, z
// segment): neighbouring blocks, which share the sites' records and edge rows,
// run on one XCD at about the same time.  (With the x group fastest the FP32
// pairs took 5.07 and 5.60 ms at 512 x 512 x 642 instead of 4.94 and 5.16, FP64
// pair 1 7.00 instead of 6.88, pair 2 the same 11.0; tiles of 4, 8 or all units
// gain no more, and all units lose the edge rows: FP64 12.0 ms.)
struct BlockPlace {
    int xg, ch, grp, seg;
};
template <typename T>
__device__ __forceinline__ BlockPlace block_place(const PairArgs<T>& a, int lb) {
    const int h = lb >> 1, xg = uniform(h % a.xgroups), rest = uniform(h / a.xgroups);
    return BlockPlace{xg, uniform(rest % a.g.nch), lb & 1, uniform(rest / a.g.nch)};
}
template <typename T, int PAIR, bool OPEN, int R>
__device__ __forceinline__ void pair_block(const PairArgs<T>& a, int lb, int wib, PairSlab<T, R, kAgain<T, PAIR>>& lds,
                                           GhostLds<T, OPEN, 1>& gl) {
    const BlockPlace p = block_place(a, lb);
    const int ch = p.ch, grp = p.grp, j0 = p.seg * a.zlen;
    const int nx = a.g.nx, j1 = min(a.g.nz, j0 + a.zlen), ib = p.xg * R;
    if (wib == 0) {   // (read after the first barriers)
        fill_table(a.g, lds.tab, ch, threadIdx.x & 63);
        gl.fill(a, ch, grp, 0);
    }
    // wave wib works on x row ib - 2 + wib; rows past either end wrap (the box
    // is periodic), and rows past the last one write nothing
    const int r = ib - 2 + wib, row = uniform(wrapi(r, nx));
    if (wib >= 2 && wib < R + 2 && r < nx) {
        pair_wave<T, PAIR, true, false, OPEN>(a, row, ch, grp, j0, j1, wib, -1, 0, lds.tab, lds.st[wib - 2], &lds,
                                              gl.get(0));
    } else {
        // the first and last two waves also load the rows beyond: -4, -3, R+2, R+3
        const bool lo = wib < 2, hi = wib >= R + 2;
        const int er = lo ? ib - 4 + wib : ib + wib;
        pair_wave<T, PAIR, false, false, OPEN>(a, row, ch, grp, j0, j1, wib, lo || hi ? uniform(wrapi(er, nx)) : -1,
                                         lo ? wib : (hi ? wib + 4 : R + 8), lds.tab, lds.st[0], &lds, gl.get(0));
    }
}

template <typename T, int PAIR, bool OPEN>
__global__ __launch_bounds__(64 * (PairShape<T, PAIR>::R + 4)) __attribute__((amdgpu_waves_per_eu(PairShape<T, PAIR>::SimdWaves)))
void k_pair(const PairArgs<T> a) {
    constexpr int R = PairShape<T, PAIR>::R;
    __shared__ PairSlab<T, R, kAgain<T, PAIR>> lds;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    __shared__ GhostLds<T, OPEN, 1> gl;
    pair_block<T, PAIR, OPEN, R>(a, xcd_remap(blockIdx.x, gridDim.x), wib, lds, gl);
}

// Many independent runs in one launch: logical block -> (run, block of run)
// from bmap; each run's arguments from the runs table (read with scalar loads).
template <typename T, int PAIR>
__global__ __launch_bounds__(64 * (PairShape<T, PAIR>::R + 4)) __attribute__((amdgpu_waves_per_eu(PairShape<T, PAIR>::SimdWaves)))
void k_pair_batch(const PairArgs<T>* __restrict__ runs, const int* __restrict__ bmap) {
    constexpr int R = PairShape<T, PAIR>::R;
    __shared__ PairSlab<T, R, kAgain<T, PAIR>> lds;
    GhostLds<T, false, 1> gl;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const __attribute__((address_space(4))) int* cm = (const __attribute__((address_space(4))) int*)bmap;
    const int run = cm[2 * lb], blk = cm[2 * lb + 1];
    const PairArgs<T> a = runs[run];   // uniform, read-only: scalar loads
    pair_block<T, PAIR, false, R>(a, blk, wib, lds, gl);
}

// The same work as a persistent kernel: a grid of resident blocks takes
// logical blocks from a work queue until it is empty.  Logical blocks keep
// the split of xcd_remap (one contiguous range per XCD, block b of the grid
// runs on XCD b % 8), and each XCD's blocks draw from their range through
// their own counter ctr[x], so neighbouring logical blocks still run on one
// XCD at about the same time.  Every block leaves the loop once its XCD's
// counter passes the range (the exit every wave reaches); the counters are
// zeroed by k_zero_ints before each launch.
template <typename T, int PAIR>
__global__ __launch_bounds__(64 * (PairShape<T, PAIR>::R + 4)) __attribute__((amdgpu_waves_per_eu(PairShape<T, PAIR>::SimdWaves)))
void k_pair_batch_q(const PairArgs<T>* __restrict__ runs, const int* __restrict__ bmap, int* __restrict__ ctr,
                    int nitems) {
    constexpr int R = PairShape<T, PAIR>::R;
    __shared__ PairSlab<T, R, kAgain<T, PAIR>> lds;
    __shared__ int next;
    GhostLds<T, false, 1> gl;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int x = blockIdx.x % 8;
    const int per = nitems / 8, rem = nitems % 8;
    const int start = x < rem ? x * (per + 1) : rem * (per + 1) + (x - rem) * per;
    const int count = per + (x < rem ? 1 : 0);
    const __attribute__((address_space(4))) int* cm = (const __attribute__((address_space(4))) int*)bmap;
    for (;;) {
        if (threadIdx.x == 0) next = atomicAdd(&ctr[x], 1);
        __syncthreads();   // (also: every wave is done with the slab of the last block)
        const int k = __builtin_amdgcn_readfirstlane(next);
        __syncthreads();   // every wave has read next before thread 0 rewrites it
        if (k >= count) break;
        const int lb = start + k;
        const int run = cm[2 * lb], blk = cm[2 * lb + 1];
        const PairArgs<T> a = runs[run];   // uniform, read-only: scalar loads
        pair_block<T, PAIR, false, R>(a, blk, wib, lds, gl);
    }
}

constexpr int kRowWaves = 4;   // waves per block of the one-row form, a unit each

template <typename T, int R>
struct LoneSlab {
    T y[2][R + 9][kF][64];   // rows -2 .. R+5 of y, and a slot idle lanes write
    SumTable tab;
    SumStage st[R + 4];
};

template <typename T, bool OPEN>
__global__ __launch_bounds__(64 * (PairShape<T, 3>::R + 4)) __attribute__((amdgpu_waves_per_eu(PairShape<T, 3>::SimdWaves)))
void k_lone(const PairArgs<T> a) {
    constexpr int R = PairShape<T, 3>::R, NW = R + 4;
    __shared__ LoneSlab<T, R> lds;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const BlockPlace p = block_place(a, xcd_remap(blockIdx.x, gridDim.x));
    const int nx = a.g.nx, ib = p.xg * NW, r = ib + wib, j0 = p.seg * a.zlen;
    if (wib == 0) fill_table(a.g, lds.tab, p.ch, threadIdx.x & 63);   // (read after the first barrier)
    const bool lo = wib < 2, hi = wib >= NW - 2;
    const int er = lo ? ib - 2 + wib : ib + wib + 2;
    lone_wave<T, false, OPEN>(a, uniform(wrapi(r, nx)), r < nx, p.ch, p.grp, j0, min(a.g.nz, j0 + a.zlen), wib,
                        lo || hi ? uniform(wrapi(er, nx)) : -1, lo ? wib : (hi ? wib + 4 : R + 8), lds.tab,
                        lds.st[wib], &lds);
}

template <typename T, bool OPEN>
__global__ __launch_bounds__(64 * kRowWaves) __attribute__((amdgpu_waves_per_eu(PairShape<T, 3>::SimdWaves)))
void k_lone_row(const PairArgs<T> a) {
    __shared__ PairRowLds<kRowWaves> lds;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int groups = (a.nunits + kRowWaves - 1) / kRowWaves;
    const int un = uniform(lb % groups) * kRowWaves + wib, j0 = uniform(lb / groups) * a.zlen;
    if (un >= a.nunits) return;
    fill_table(a.g, lds.tab[wib], un >> 1, threadIdx.x & 63);
    lone_wave<T, true, OPEN>(a, 0, true, un >> 1, un & 1, j0, min(a.g.nz, j0 + a.zlen), 0, -1, 0, lds.tab[wib], lds.st[wib],
                       (LoneSlab<T, 1>*)nullptr);
}

template <typename T, int PAIR, bool OPEN>
__global__ __launch_bounds__(64 * kRowWaves) __attribute__((amdgpu_waves_per_eu(PairShape<T, PAIR>::SimdWaves)))
void k_pair_row(const PairArgs<T> a) {
    __shared__ PairRowLds<kRowWaves> lds;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lb = xcd_remap(blockIdx.x, gridDim.x);
    const int groups = (a.nunits + kRowWaves - 1) / kRowWaves;
    const int un = uniform(lb % groups) * kRowWaves + wib, j0 = uniform(lb / groups) * a.zlen;
    if (un >= a.nunits) return;
    fill_table(a.g, lds.tab[wib], un >> 1, threadIdx.x & 63);   // (the wave's own: its LDS accesses stay in order)
    __shared__ GhostLds<T, OPEN, kRowWaves> gl;
    gl.fill(a, un >> 1, un & 1, wib);
    pair_wave<T, PAIR, true, true, OPEN>(a, 0, un >> 1, un & 1, j0, min(a.g.nz, j0 + a.zlen), 0, -1, 0, lds.tab[wib],
                                   lds.st[wib], (PairRowLds<kRowWaves>*)nullptr, gl.get(wib));
}

// ---------------------------------------------------------------------------
// partial sums of a state (after init, upload or renormalisation): a wave per
// unit and run of sites
// ---------------------------------------------------------------------------
constexpr int kSumSites = 16;   // sites per wave

template <typename T>
__global__ __launch_bounds__(256) void k_pair_sums(const Geometry g, const T* __restrict__ y, double* __restrict__ part) {
    __shared__ PairRowLds<4> lds;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const long long nsites = (long long)g.nx * g.nz, runs = (nsites + kSumSites - 1) / kSumSites;
    const long long id = (long long)blockIdx.x * 4 + wib;
    const int nu = 2 * g.nch;
    if (id >= runs * nu) return;
    const int un = (int)(id % nu), ch = un >> 1, grp = un & 1;
    fill_table(g, lds.tab[wib], ch, lane);
    const int pv = min(ch * 64 + lane, g.nv - 1);
    const long long s0 = id / nu * kSumSites, s1 = min(nsites, s0 + kSumSites);
    const unsigned vrec = sum_offset(lane, kRec * 8);
    for (long long s = s0; s < s1; ++s) {
        const T* p = y + site_off(g, s) + (long long)(grp * kF) * g.nvp + pv;
        const double ee = p[0], mm = p[g.nvp], emr = p[2 * (long long)g.nvp], emi = p[3 * (long long)g.nvp];
        direction_sums(emr, emi, ee - mm, lds.st[wib], lds.tab[wib], lane,
                       prs((unsigned long long)(part + (s * g.nch + ch) * kPairRec + grp * kRec), kRec * 8), vrec, 0);
    }
}

// ---------------------------------------------------------------------------
// totals of a site's partial sums in chunk order, and the moments they give.
// Totals are stored as the combinations the moments are made of, per monomial
//   D = (bemr - emr, bemi + emi, (bee - bmm) - (ee - mm))   [site][kMono][3]
//   Q = (bemr + emr, bemi - emi, (bee - bmm) + (ee - mm))   after all D's
// ---------------------------------------------------------------------------
template <bool COMP>
__device__ __forceinline__ double chunk_sum(const double* __restrict__ rec, int nch) {
    double sum = rec[0], err = 0.0;
#pragma unroll 4
    for (int c = 1; c < nch; ++c) {
        const double x = rec[(long long)c * kPairRec];
        if constexpr (COMP) {   // (FP32 form: as k_moment_totals)
            const double s = sum + x, bb = s - sum;
            err += (sum - (s - bb)) + (x - bb);
            sum = s;
        } else {
            sum += x;
        }
    }
    return sum + err;
}
// Open z: the two ghost sites past each end of the stencil input y, and their
// partial direction sums (which the prediction adds).  A wave per (x row, end,
// depth) and chunk: at 1 x 4096 x 642 it is the latency of one wave's work (a
// block per site, its waves sharing the chunks, took 24 us).  The waves are
// numbered through: with blocks of four chunks of one site, three of four waves
// idle at 12-42 directions, a step took 529 us instead of 375 at 4096 x 12 x 12
// and 354 instead of 283 at 2048 x 16 x 42 (FP32).  The waves of row 0 also write
// the inflow values the inner input has there (gin: they are the same in every
// x row).
constexpr int kGhostWaves = 4;
struct OpenArgs {
    unsigned long long y;             // u, Y3 or u2
    const double *G0, *G0b, *t_dev;
    Inflow in;
    double cdt, cdt_inner;            // times of y and of the inner input, from t_dev
    double* part;                     // records [nx][end][depth][chunk]
    unsigned long long gin;
};
template <typename T>
__global__ __launch_bounds__(64 * kGhostWaves) void k_pair_ghosts(const Geometry g, const OpenArgs a) {
    __shared__ PairRowLds<kGhostWaves> lds;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int id = uniform((int)blockIdx.x * kGhostWaves + wib), site = uniform(id / g.nch), ch = uniform(id % g.nch);
    if (site >= 4 * g.nx) return;
    const int i = site / 4, end = site / 2 % 2, depth = site % 2 + 1;
    const int j = end == 0 ? -depth : g.nz - 1 + depth, e0 = end == 0 ? 0 : g.nz - 1;
    T* const y = (T*)a.y;
    fill_table(g, lds.tab[wib], ch, lane);
    const unsigned vrec = sum_offset(lane, kRec * 8);
    const long long dz = end == 0 ? g.srec : -g.srec;
    const int pv = min(ch * 64 + lane, g.nv - 1);
    const double vz = g.vz[pv];
    const bool in = end == 0 ? vz > 0.0 : vz < 0.0;
#pragma unroll
    for (int grp = 0; grp < 2; ++grp) {
        double h[kF], x[kF];
        T* const p = y + elem_off(g, i, j + g.zoff, grp * kF) + pv;
        const T* const e = y + elem_off(g, i, e0 + g.zoff, grp * kF) + pv;
        const double hg = 0.5 * (grp ? a.G0b : a.G0)[pv];
        if (in) open_inflow(a.in, vz, j, a.t_dev[0] + a.cdt, hg, h);
#pragma unroll
        for (int f = 0; f < kF; ++f) {
            const long long o = (long long)f * g.nvp;
            const T v = in ? (T)h[f] : (T)open_extrapolate(depth, (double)e[o], (double)e[o + dz], (double)e[o + 2 * dz]);
            if (ch * 64 + lane < g.nv) p[o] = v;
            x[f] = (double)v;
        }
        direction_sums(x[2], x[3], x[0] - x[1], lds.st[wib], lds.tab[wib], lane,
                       prs((unsigned long long)(a.part + ((long long)site * g.nch + ch) * kPairRec + grp * kRec), kRec * 8),
                       vrec, 0);
        if (i == 0 && in) {
            T* const q = (T*)a.gin + (long long)((end * 2 + depth - 1) * kNVar + grp * kF) * g.nvp + pv;
            open_inflow(a.in, vz, j, a.t_dev[0] + a.cdt_inner, hg, h);
#pragma unroll
            for (int f = 0; f < kF; ++f) q[(long long)f * g.nvp] = (T)h[f];
        }
    }
}
// A block adds the records of kTotSites sites, a thread per sum (the reads are
// the whole pass: 1.25 GB at 512 x 512 x 642), and combines them through LDS.
constexpr int kTotSites = 8, kTotThreads = 448;
static_assert(kTotSites * kPairRec <= kTotThreads, "a thread per sum");
template <bool COMP>
__device__ __forceinline__ void pair_totals_body(const double* __restrict__ part, int nch, long long nsites,
                                                 double* __restrict__ tot, long long blk, double (&sums)[kTotSites * kPairRec]) {
    const long long s0 = blk * kTotSites;
    const int n = (int)min((long long)kTotSites, nsites - s0), tid = threadIdx.x;
    if (tid < n * kPairRec)
        sums[tid] = chunk_sum<COMP>(part + (s0 + tid / kPairRec) * nch * kPairRec + tid % kPairRec, nch);
    __syncthreads();
    if (tid < n * kPairRec) {
        const int k = tid < n * kRec ? tid : tid - n * kRec;   // entry of D, then of Q
        const double nu = sums[k / kRec * kPairRec + k % kRec], bar = sums[k / kRec * kPairRec + kRec + k % kRec];
        const bool plus = (k % 3 == 1) == (tid < n * kRec);
        tot[(tid < n * kRec ? 0 : nsites * kRec) + s0 * kRec + k] = plus ? bar + nu : bar - nu;
    }
}

struct PredictArgs {
    const double* tot;    // D, then Q
    const double* base;   // what the prediction starts from (an m, or null: that of tot's state)
    double* m;            // record of tot's state: mu times its moments, with the vacuum terms
    double* inner;        // the same of base + c k (null: not wanted)
    const double* gpart;  // open z: records of the two ghost sites at each end, [nx][end][depth][chunk] (null: periodic)
    int nch;
    double c;
    double mu, mu2, p2st, p2ct, pmo, ct2, st;
    double twelve_dx, twelve_dz, ko_x, ko_z;
    int nx, nz;
};

// A block predicts kPredZ sites of one x row, 16 threads a site: thread
// (site, s) moment component a = s % 4 of vector s / 4 (A: bemr - emr,
// B: bemi + emi, C: bee - bmm - ee + mm).  The totals it needs (the row's
// sites and two more at each end, the same sites of the four neighbouring
// rows) are staged in LDS with coalesced loads: read from L2 by each thread
// where needed, the pass took 0.29 ms at 512 x 512, a third of it index
// arithmetic.  The moments of k follow nuosc_class.cpp:115-287 summed over
// directions with w u_a.
constexpr int kPredZ = 16;
struct PredictLds {
    double d[kPredZ + 4][kRec];       // own row, z - 2 .. z + 17
    double x[4][kPredZ][kRec];        // x - 2, x - 1, x + 1, x + 2
    double q[kPredZ][kRec];
};
// monomial of u_a u_b, a <= b (0: yy, which is 1 - xx - zz)
__device__ __forceinline__ int mono_of(int lo, int hi) { return lo == 0 ? hi : (lo == 1 ? 3 + hi : 5 + lo); }
__device__ __forceinline__ double second(const double* t, int a, int b, int c) {
    if (a == 2 && b == 2) return t[c] - t[4 * 3 + c] - t[8 * 3 + c];
    return t[mono_of(min(a, b), max(a, b)) * 3 + c];
}

// blocks of one run
__host__ __device__ inline long long predict_blocks(int nx, int nz) { return (long long)nx * ((nz + kPredZ - 1) / kPredZ); }

__device__ __forceinline__ void predict_body(const PredictArgs& p, int blk, PredictLds& l) {
    const int tiles = (p.nz + kPredZ - 1) / kPredZ;
    const int i = blk / tiles, z0 = (blk % tiles) * kPredZ, nz = p.nz;
    const int n = min(kPredZ, nz - z0), tid = threadIdx.x;
    const long long row = (long long)i * nz, nsites = (long long)p.nx * nz;
    // (all loads ahead of the first LDS store: in loops, each waiting for its own,
    // the kernel took 8.2 us at 20 x 200 sites instead of 5.4, and 98 us at 512 x
    // 512 instead of 60)
    constexpr int kD = ((kPredZ + 4) * kRec + 255) / 256, kX = (kPredZ * kRec + 255) / 256;
    double rd[kD], rx[4][kX], rq[kX];
#pragma unroll
    for (int m = 0; m < kD; ++m) {
        const int k = min(tid + 256 * m, (n + 4) * kRec - 1), z = z0 - 2 + k / kRec;
        rd[m] = p.tot[(row + wrapi(z, nz)) * kRec + k % kRec];
        if (p.gpart && (z < 0 || z >= nz)) {
            const double* t = p.gpart + (i * 4ll + (z < 0 ? -1 - z : 2 + z - nz)) * p.nch * kPairRec + k % kRec;
            const double nu = chunk_sum<true>(t, p.nch), bar = chunk_sum<true>(t + kRec, p.nch);
            rd[m] = k % kRec % 3 == 1 ? bar + nu : bar - nu;
        }
    }
#pragma unroll
    for (int m = 0; m < kX; ++m) {
        const int k = min(tid + 256 * m, n * kRec - 1);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            rx[q][m] = p.tot[((long long)wrapi(i + (q < 2 ? q - 2 : q - 1), p.nx) * nz + z0) * kRec + k];
        rq[m] = p.tot[(nsites + row + z0) * kRec + k];
    }
    // (threads past the end store the last entry again)
#pragma unroll
    for (int m = 0; m < kD; ++m) (&l.d[0][0])[min(tid + 256 * m, (n + 4) * kRec - 1)] = rd[m];
#pragma unroll
    for (int m = 0; m < kX; ++m) {
        const int k = min(tid + 256 * m, n * kRec - 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) (&l.x[q][0][0])[k] = rx[q][m];
        (&l.q[0][0])[k] = rq[m];
    }
    __syncthreads();
    const int zl = tid / kMomStride, s = tid % kMomStride;
    if (zl >= n) return;
    const long long o = (row + z0 + zl) * kMomStride + s;
    if (s >= kNMom) {
        p.m[o] = 0.0;
        if (p.inner) p.inner[o] = 0.0;
        return;
    }
    const int a = s & 3, v = s >> 2;
    const double *d = l.d[zl + 2], *q = l.q[zl];
    const double m0 = d[a * 3 + v];
    // (the record's offset: see precession())
    const double mm = p.mu * m0 + (s == 0 ? -p.pmo * p.st : (s == 8 ? p.p2ct : 0.0));
    p.m[o] = mm;
    if (!p.inner) return;
    // transport: advection multiplies by vx or vz, Kreiss-Oliger by nothing
    double kt = 0.0;
#pragma unroll
    for (int ax = 0; ax < 2; ++ax) {
        const int b = ax ? 3 : 1, second_ab = mono_of(min(a, b), max(a, b)) * 3 + v, first = a * 3 + v;
        auto at = [&](int k) { return ax ? l.d[zl + (k < 2 ? k : k + 1)] : l.x[k][zl]; };
        const double adv = (at(0)[second_ab] - at(3)[second_ab]) - 8.0 * (at(1)[second_ab] - at(2)[second_ab]);
        const double ko = at(0)[first] + at(3)[first] - 4 * (at(1)[first] + at(2)[first]) + 6 * m0;
        kt += (ax ? p.ko_z : p.ko_x) * ko - adv / (ax ? p.twelve_dz : p.twelve_dx);
    }
    // interaction: sum over b of s_b (moment b) (second moment a b), s = (1, -1, -1, -1)
    double loc = 0.0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const double Ab = d[b * 3], Bb = d[b * 3 + 1], Cb = d[b * 3 + 2];
        double x;
        if (v == 0)        // k_emr of bar minus nu: -mu [ d3 B + (bemi - emi) C ]
            x = -p.mu * (second(d, a, b, 2) * Bb + Cb * second(q, a, b, 1));
        else if (v == 1)   // k_emi of bar plus nu: mu [ -(bee - bmm + ee - mm) A + (bemr + emr) C ]
            x = p.mu * (Cb * second(q, a, b, 0) - second(q, a, b, 2) * Ab);
        else               // k_ee - k_mm = 2 k_ee: 2 mu2 [ (bemi - emi) A + (bemr - emr) B ]
            x = 2 * p.mu2 * (second(q, a, b, 1) * Ab + second(d, a, b, 0) * Bb);
        loc += b == 0 ? x : -x;
    }
    const double r1 = q[a * 3], i1 = q[a * 3 + 1], e1 = q[a * 3 + 2];
    const double vac = v == 0 ? -p.p2ct * i1 : (v == 1 ? p.pmo * (p.ct2 * r1 + p.st * e1) : -2 * p.p2st * i1);
    p.inner[o] = (p.base ? p.base[o] : mm) + p.mu * (p.c * (loc + kt + vac));
}

template <bool COMP>
__global__ __launch_bounds__(kTotThreads) void k_pair_totals(const double* __restrict__ part, int nch, long long nsites,
                                                             double* __restrict__ tot) {
    __shared__ double sums[kTotSites * kPairRec];
    pair_totals_body<COMP>(part, nch, nsites, tot, blockIdx.x, sums);
}
__global__ __launch_bounds__(256) void k_pair_predict(const PredictArgs p) {
    __shared__ PredictLds lds;
    predict_body(p, blockIdx.x, lds);
}

struct SumArgs {
    const double* part;
    double* tot;
    int nch;
    long long nsites;
};
template <bool COMP>
__global__ __launch_bounds__(kTotThreads) void k_pair_totals_batch(const SumArgs* __restrict__ runs, const int* __restrict__ map) {
    const __attribute__((address_space(4))) int* cm = (const __attribute__((address_space(4))) int*)map;
    const SumArgs a = runs[cm[2 * blockIdx.x]];
    __shared__ double sums[kTotSites * kPairRec];
    pair_totals_body<COMP>(a.part, a.nch, a.nsites, a.tot, cm[2 * blockIdx.x + 1], sums);
}
__global__ __launch_bounds__(256) void k_pair_predict_batch(const PredictArgs* __restrict__ runs, const int* __restrict__ map) {
    const __attribute__((address_space(4))) int* cm = (const __attribute__((address_space(4))) int*)map;
    __shared__ PredictLds lds;
    const PredictArgs p = runs[cm[2 * blockIdx.x]];
    predict_body(p, cm[2 * blockIdx.x + 1], lds);
}

// x rows a block of a pair (or of the lone stage) writes
int pair_rows(int esize, int pair) {
    if (esize == 4) return PairShape<float, 1>::R + (pair == kLone ? 4 : 0);
    return pair == 2 ? PairShape<double, 2>::R : PairShape<double, 1>::R + (pair == kLone ? 4 : 0);
}

template <typename T>
PairArgs<T> pair_args(const Geometry& g, const Physics& ph, int zlen, int pair, const PairBuffers& b, double dt) {
    PairArgs<T> a{};
    a.g = g;
    const bool first = pair == 1 || pair == 3;   // u is the stencil input
    a.y = (unsigned long long)(first ? b.u : b.y3);
    a.u = (unsigned long long)b.u;
    a.a = (unsigned long long)b.a;
    a.out = (unsigned long long)(first ? b.y3 : b.unew);
    a.m1 = (unsigned long long)(first ? b.mu : b.m3);
    a.m2 = (unsigned long long)b.min;
    a.m0 = (unsigned long long)b.mu;
    a.part = (unsigned long long)b.part;
    a.gin = (unsigned long long)b.gin;
    switch (pair) {
        case 1: a.c1 = a.c2 = 0.5 * dt; a.cA = dt; break;
        case 2: a.c1 = dt; a.c2 = 1.0 / 6.0 * dt; break;
        case 3: a.c1 = dt; a.c2 = 3.0 / 4.0; a.cA = 1.0 / 4.0; break;
        default: a.c1 = dt; a.c2 = 1.0 / 3.0; a.cA = 2.0 / 3.0; break;
    }
    a.zlen = zlen;
    const int rows = pair_rows(sizeof(T), pair);
    a.xgroups = g.nx == 1 ? 1 : (g.nx + rows - 1) / rows;
    a.nunits = 2 * g.nch;
    return a;
}

PredictArgs predict_args(const Geometry& g, const Physics& ph, int pair, const PairBuffers& b, double dt) {
    PredictArgs p{};
    p.tot = b.tot;
    p.base = pair == 2 ? b.mu : nullptr;
    p.m = pair == 1 || pair == 3 ? b.mu : b.m3;
    p.inner = pair == kLone ? nullptr : b.min;
    p.gpart = g.bc ? b.gpart : nullptr;
    p.nch = g.nch;
    p.c = pair == 1 ? 0.5 * dt : dt;
    p.mu = ph.mu;
    p.mu2 = 2 * ph.mu;
    p.p2st = ph.pmo * 2 * ph.st;
    p.p2ct = ph.pmo * 2 * ph.ct;
    p.pmo = ph.pmo;
    p.ct2 = 2 * ph.ct;
    p.st = ph.st;
    p.twelve_dx = g.twelve_dx;
    p.twelve_dz = g.twelve_dz;
    p.ko_x = g.ko_x;
    p.ko_z = g.ko_z;
    p.nx = g.nx;
    p.nz = g.nz;
    return p;
}

}  // namespace

bool pair_capable(const Geometry& g) {
    return g.nf == kNVar && (g.bc == 0 || (g.zoff >= 2 && g.nz >= 3)) && !g.ko5 && g.adv == kAdvCfd4;
}

namespace {
// blocks of the box form (batches take it for one-row grids too)
long long pair_box_blocks(const Geometry& g, int esize, int pair, int zlen) {
    const int R = pair_rows(esize, pair);
    return (long long)((g.nz + zlen - 1) / zlen) * 2 * g.nch * ((g.nx + R - 1) / R);
}
long long pair_blocks(const Geometry& g, int esize, int pair, int zlen) {
    if (g.nx > 1) return pair_box_blocks(g, esize, pair, zlen);
    return (g.nz + zlen - 1) / zlen * ((2 * g.nch + kRowWaves - 1) / kRowWaves);
}

// Time of a pair kernel's blocks in steps of the z march: rounds of as many
// blocks as the GPU holds at once (one per CU in the box form, counted as
// three in the one-row form, of which FP32 holds five: 3001 x 492 in FP32 takes
// 110-113 us in segments of 24 or 16 sites, 130 in 10), each of zlen steps and
// about eight more: four that write nothing, the rest the block's start.  At
// 512 x 512 x 642 the model orders segments of 64 .. 512 sites as they measure
// in both precisions; 20 x 200 x 162: segments of 13 sites are two rounds
// (75 us a kernel), 15 one.
double pair_march_steps(long long blocks, int zlen, bool one_row, int num_cus) {
    const long long slots = (long long)num_cus * (one_row ? 3 : 1);
    return (double)((blocks + slots - 1) / slots) * (zlen + 8);
}
}  // namespace

int pair_waves(const Geometry& g, int esize, int zlen) {
    return (int)(pair_blocks(g, esize, 1, zlen) * (g.nx == 1 ? kRowWaves : pair_rows(esize, 1) + 4));
}

// (Each kernel its own: they differ in the rows of a block, and so in the blocks
// of a segment.  With one length for both pairs, and that for SSP-RK3 too, a step
// of 20 x 200 x 162 took 138 us instead of 125, 203 x 157 x 362 1.37 ms instead of
// 1.32, SSP-RK3 on 46 x 78 x 92 105 us instead of 69.)
int plan_pair_zlen(const Geometry& g, int esize, int pair, int num_cus) {
    int best = g.nz;
    double least = 1e300;
    for (int most = std::min(g.nz, 1024); most >= 1; --most) {
        const int nseg = (g.nz + most - 1) / most, zlen = (g.nz + nseg - 1) / nseg;   // equal segments
        const double t = pair_march_steps(pair_blocks(g, esize, pair, zlen), zlen, g.nx == 1, num_cus);
        if (t < least) {
            least = t;
            best = zlen;
        }
    }
    return best;
}

int plan_batch_zlen(const std::vector<Geometry>& gs, int esize, int num_cus) {
    int best = 64;
    double least = 1e300;
    for (int zlen : {4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256}) {
        double t = 0.0;
        for (int pair : {1, 2}) {
            long long blocks = 0;
            for (const Geometry& g : gs) blocks += pair_box_blocks(g, esize, pair, std::min(zlen, g.nz));
            t += pair_march_steps(blocks, zlen, false, num_cus);
        }
        if (t < least) {
            least = t;
            best = zlen;
        }
    }
    return best;
}

namespace {
template <typename T, bool OPEN>
void launch_pair_form(int pair, const PairArgs<T>& a, unsigned nseg, hipStream_t s) {
    if (a.g.nx == 1) {
        const dim3 grid(nseg * ((a.nunits + kRowWaves - 1) / kRowWaves)), block(64 * kRowWaves);
        if (pair == 1) hipLaunchKernelGGL((k_pair_row<T, 1, OPEN>), grid, block, 0, s, a);
        else if (pair == 2) hipLaunchKernelGGL((k_pair_row<T, 2, OPEN>), grid, block, 0, s, a);
        else if (pair == 3) hipLaunchKernelGGL((k_pair_row<T, 3, OPEN>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_lone_row<T, OPEN>), grid, block, 0, s, a);
    } else {
        const dim3 grid(nseg * (unsigned)(a.xgroups * a.nunits));
        const dim3 block(64 * (pair_rows(sizeof(T), pair) + (pair == kLone ? 0 : 4)));
        if (pair == 1) hipLaunchKernelGGL((k_pair<T, 1, OPEN>), grid, block, 0, s, a);
        else if (pair == 2) hipLaunchKernelGGL((k_pair<T, 2, OPEN>), grid, block, 0, s, a);
        else if (pair == 3) hipLaunchKernelGGL((k_pair<T, 3, OPEN>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((k_lone<T, OPEN>), grid, block, 0, s, a);
    }
}
}  // namespace

template <typename T>
hipError_t launch_pair(int pair, const Geometry& g, const Physics& ph, int zlen, const PairBuffers& b, double dt,
                       hipStream_t s) {
    if (!pair_capable(g) || zlen < 1 || g.lpr != 64) return hipErrorInvalidValue;
    const PairArgs<T> a = pair_args<T>(g, ph, zlen, pair, b, dt);
    const unsigned nseg = (unsigned)((g.nz + zlen - 1) / zlen);
    if (g.bc) launch_pair_form<T, true>(pair, a, nseg, s);
    else launch_pair_form<T, false>(pair, a, nseg, s);
    return hipGetLastError();
}

hipError_t launch_pair_predict(int pair, const Geometry& g, const Physics& ph, const PairBuffers& b, double dt,
                               hipStream_t s) {
    const PredictArgs p = predict_args(g, ph, pair, b, dt);
    hipLaunchKernelGGL(k_pair_predict, dim3((unsigned)predict_blocks(g.nx, g.nz)), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_pair_totals(const Geometry& g, bool compensated, const PairBuffers& b, hipStream_t s) {
    const long long nsites = (long long)g.nx * g.nz;
    const dim3 grid((unsigned)((nsites + kTotSites - 1) / kTotSites));
    if (compensated) hipLaunchKernelGGL((k_pair_totals<true>), grid, dim3(kTotThreads), 0, s, b.part, g.nch, nsites, b.tot);
    else hipLaunchKernelGGL((k_pair_totals<false>), grid, dim3(kTotThreads), 0, s, b.part, g.nch, nsites, b.tot);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_pair_ghosts(int pair, const Geometry& g, const PairBuffers& b, const double* G0, const double* G0b,
                              const Inflow& in, const double* t_dev, double dt, hipStream_t s) {
    if (!pair_capable(g)) return hipErrorInvalidValue;
    const bool first = pair == 1 || pair == 3;
    const OpenArgs a{(unsigned long long)(first ? b.u : b.y3), G0, G0b, t_dev, in, first ? 0.0 : 0.5 * dt,
                     pair == 1 ? 0.5 * dt : dt, b.gpart, (unsigned long long)b.gin};
    const long long waves = 4ll * g.nx * g.nch;
    const dim3 grid((unsigned)((waves + kGhostWaves - 1) / kGhostWaves));
    hipLaunchKernelGGL((k_pair_ghosts<T>), grid, dim3(64 * kGhostWaves), 0, s, g, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_pair_sums(const Geometry& g, const T* y, double* part, hipStream_t s) {
    const long long runs = ((long long)g.nx * g.nz + kSumSites - 1) / kSumSites;
    hipLaunchKernelGGL((k_pair_sums<T>), dim3((unsigned)((runs * 2 * g.nch + 3) / 4)), dim3(256), 0, s, g, y, part);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// batched runs: the launches of a step for every member run; the runs keep
// their own buffers, segments and physics.  All tables live in one device
// buffer, [pairs 1, 2] x [flips 0, 1] of arguments and the block maps, and a
// rebuild (a member joins or leaves) reuses it.
// ---------------------------------------------------------------------------
namespace {

template <typename T>
hipError_t batch_build_t(BatchTables& t, const std::vector<BatchMember>& ms, hipStream_t s) {
    const int n = (int)ms.size();
    TableImage im;
    // blocks of the two pairs, the totals and the prediction -> (member, block of member)
    std::vector<long long> count[4];
    for (const BatchMember& m : ms) {
        const Geometry& g = m.g;
        const long long sites = (long long)g.nx * g.nz;
        // (the box form for every member, one-row grids included)
        for (int pair : {1, 2}) count[pair - 1].push_back(pair_box_blocks(g, sizeof(T), pair, m.zlen[pair - 1]));
        count[2].push_back((sites + kTotSites - 1) / kTotSites);
        count[3].push_back(predict_blocks(g.nx, g.nz));
    }
    size_t off_args[2][2], off_pre[2][2], off_map[4];
    for (int flip = 0; flip < 2; ++flip)
        for (int pair = 1; pair <= 2; ++pair) {
            std::vector<PairArgs<T>> pa(n);
            std::vector<PredictArgs> pp(n);
            for (int r = 0; r < n; ++r) {
                PairBuffers b = ms[r].b;
                if (flip) {
                    const void* u = b.u;
                    b.u = b.unew;
                    b.unew = const_cast<void*>(u);
                }
                pa[r] = pair_args<T>(ms[r].g, ms[r].ph, ms[r].zlen[pair - 1], pair, b, ms[r].dt);
                pp[r] = predict_args(ms[r].g, ms[r].ph, pair, b, ms[r].dt);
            }
            off_args[pair - 1][flip] = im.put(pa.data(), n * sizeof(PairArgs<T>));
            off_pre[pair - 1][flip] = im.put(pp.data(), n * sizeof(PredictArgs));
        }
    std::vector<SumArgs> sa(n);
    for (int r = 0; r < n; ++r)
        sa[r] = SumArgs{ms[r].b.part, ms[r].b.tot, ms[r].g.nch, (long long)ms[r].g.nx * ms[r].g.nz};
    const size_t off_sum = im.put(sa.data(), n * sizeof(SumArgs));
    int blocks[4];
    for (int k = 0; k < 4; ++k) off_map[k] = im.put_map(count[k], blocks[k]);
    const std::vector<int> zeros(kBatchCounters, 0);
    const size_t off_ctr = im.put(zeros.data(), kBatchCounters * sizeof(int));
    hipError_t e = im.upload(t.buf, t.bytes, s);
    if (e != hipSuccess) return e;
    // persistent launch: a grid of as many blocks as the GPU holds at once
    e = resident_blocks((const void*)k_pair_batch_q<T, 1>, 64 * (PairShape<T, 1>::R + 4), t.pgrid[0]);
    if (e != hipSuccess) return e;
    e = resident_blocks((const void*)k_pair_batch_q<T, 2>, 64 * (PairShape<T, 2>::R + 4), t.pgrid[1]);
    if (e != hipSuccess) return e;
    char* d = static_cast<char*>(t.buf);
    for (int p = 0; p < 2; ++p)
        for (int flip = 0; flip < 2; ++flip) {
            t.args[p][flip] = d + off_args[p][flip];
            t.pre[p][flip] = d + off_pre[p][flip];
        }
    t.sum = d + off_sum;
    for (int p = 0; p < 2; ++p) {
        t.bmap[p] = (int*)(d + off_map[p]);
        t.nblocks[p] = blocks[p];
    }
    t.tmap = (int*)(d + off_map[2]);
    t.pmap = (int*)(d + off_map[3]);
    t.ctr = (int*)(d + off_ctr);
    t.tblocks = blocks[2];
    t.pblocks = blocks[3];
    return hipSuccess;
}

template <typename T, int PAIR>
hipError_t batch_pair_t(const BatchTables& t, int flip, hipStream_t s) {
    const dim3 block(64 * (PairShape<T, PAIR>::R + 4));
    const PairArgs<T>* a = (const PairArgs<T>*)t.args[PAIR - 1][flip];
    const int n = t.nblocks[PAIR - 1];
    if (t.launch == kBatchPersistent) {
        int* c = t.ctr + 8 * (PAIR - 1);
        const hipError_t e = launch_zero_ints(c, 8, s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL((k_pair_batch_q<T, PAIR>), dim3(t.pgrid[PAIR - 1]), block, 0, s, a, t.bmap[PAIR - 1], c, n);
    } else {
        hipLaunchKernelGGL((k_pair_batch<T, PAIR>), dim3(n), block, 0, s, a, t.bmap[PAIR - 1]);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t batch_build(BatchTables& t, const std::vector<BatchMember>& ms, int esize, int launch, hipStream_t s) {
    t.esize = esize;
    t.launch = launch;
    t.nblocks[0] = t.nblocks[1] = 0;
    if (ms.empty()) return hipSuccess;
    for (const auto& m : ms)
        if (!pair_capable(m.g) || m.zlen[0] < 1 || m.zlen[1] < 1 || m.g.lpr != 64) return hipErrorInvalidValue;
    return esize == 8 ? batch_build_t<double>(t, ms, s) : batch_build_t<float>(t, ms, s);
}

void batch_free(BatchTables& t) {
    if (t.buf) (void)hipFree(t.buf);
    t.buf = nullptr;
    t.bytes = 0;
    t.nblocks[0] = t.nblocks[1] = 0;
}

hipError_t batch_pair(const BatchTables& t, int pair, int flip, hipStream_t s) {
    if (t.nblocks[0] == 0) return hipSuccess;
    if (t.esize == 8) return pair == 1 ? batch_pair_t<double, 1>(t, flip, s) : batch_pair_t<double, 2>(t, flip, s);
    return pair == 1 ? batch_pair_t<float, 1>(t, flip, s) : batch_pair_t<float, 2>(t, flip, s);
}

hipError_t batch_step(const BatchTables& t, int flip, hipStream_t s) {
    if (t.nblocks[0] == 0) return hipSuccess;
    for (int pair = 1; pair <= 2; ++pair) {
        hipLaunchKernelGGL(k_pair_predict_batch, dim3(t.pblocks), dim3(256), 0, s,
                           (const PredictArgs*)t.pre[pair - 1][flip], t.pmap);
        const hipError_t e = batch_pair(t, pair, flip, s);
        if (e != hipSuccess) return e;
        const dim3 tg(t.tblocks), tb(kTotThreads);
        if (t.esize == 4) hipLaunchKernelGGL((k_pair_totals_batch<true>), tg, tb, 0, s, (const SumArgs*)t.sum, t.tmap);
        else hipLaunchKernelGGL((k_pair_totals_batch<false>), tg, tb, 0, s, (const SumArgs*)t.sum, t.tmap);
    }
    return hipGetLastError();
}

#define NUOSC_PAIR_INST(T)                                                                                        \
    template hipError_t launch_pair<T>(int, const Geometry&, const Physics&, int, const PairBuffers&, double,     \
                                       hipStream_t);                                                              \
    template hipError_t launch_pair_ghosts<T>(int, const Geometry&, const PairBuffers&, const double*, const double*, \
                                              const Inflow&, const double*, double, hipStream_t);                 \
    template hipError_t launch_pair_sums<T>(const Geometry&, const T*, double*, hipStream_t);
NUOSC_PAIR_INST(double)
NUOSC_PAIR_INST(float)
#undef NUOSC_PAIR_INST

}  // namespace nuosc
