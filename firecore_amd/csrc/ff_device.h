// FP32 device force-field terms of the multi-system MMFF relaxation.
//
// Each function restates one term of the reference CPU force field in single
// precision for gfx950; the reference line ranges are given per function.
// The same functions serve the split kernels (one launch per phase) and the
// persistent relaxation kernel (all phases in one workgroup).
#pragma once
#include <hip/hip_runtime.h>

namespace fcd {

constexpr float COULOMB_K = 14.3996448915f;  // eV*A/e^2 (cpp/common/constants.h:9)

struct V3 {
    float x, y, z;
};
__device__ __forceinline__ V3 mk(float x, float y, float z) { return V3{x, y, z}; }
__device__ __forceinline__ V3 xyz(const float4& a) { return V3{a.x, a.y, a.z}; }
__device__ __forceinline__ V3 operator+(V3 a, V3 b) { return V3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ V3 operator-(V3 a, V3 b) { return V3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ V3 operator*(V3 a, float s) { return V3{a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ void operator+=(V3& a, V3 b) { a.x += b.x; a.y += b.y; a.z += b.z; }
__device__ __forceinline__ void operator-=(V3& a, V3 b) { a.x -= b.x; a.y -= b.y; a.z -= b.z; }
__device__ __forceinline__ float dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ V3 zero3() { return V3{0.f, 0.f, 0.f}; }
__device__ __forceinline__ V3 cross(V3 a, V3 b) {
    return V3{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// The thread index as a value that the compiler cannot see through.  It hoists
// whatever derives from threadIdx.x (LDS and global addresses, masks, unpacked
// neighbour lists) out of the relaxation kernel's loops and then spills it: with an
// index of its own per system, segment and step the kernel needs 30 registers fewer.
__device__ __forceinline__ int opaque_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// Gives v some value without an instruction.  A variable that is set on some paths
// only counts as carried from iteration to iteration, and holds its registers all
// the time; set to anything on the other paths it does not.
__device__ __forceinline__ void any_value(float4& v) {
    asm volatile("" : "=v"(v.x), "=v"(v.y), "=v"(v.z), "=v"(v.w));
}

// Wave shift by one lane (DPP wave_shl:1 with bound_ctrl): lane l receives
// lane l+1's value, lane 63 receives 0.  Needs all 64 lanes active.
__device__ __forceinline__ float dpp_shl1_zero(float src) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, src), 0x130, 0xF, 0xF,
                                                                 true));
}

// Stores v at LDS byte address `addr` + off (off a constant) from lane 0 alone, if it is
// active.  Narrowing exec for one instruction costs two scalar ones; the branch the compiler
// makes of `if (lane == 0)` costs six and splits the block, so nothing is scheduled across
// it.  exec comes back as it was.
typedef float f32x3 __attribute__((ext_vector_type(3)));
#define lane0_store(addr, off, v)                                                                               \
    do {                                                                                                        \
        unsigned long long saved_;                                                                              \
        asm volatile("s_and_saveexec_b64 %0, 1\n\tds_write_b96 %1, %2 offset:%3\n\ts_mov_b64 exec, %0"          \
                     : "=&s"(saved_)                                                                            \
                     : "v"(addr), "v"(f32x3{(v).x, (v).y, (v).z}), "n"(off)                                     \
                     : "memory", "scc");                                                                        \
    } while (0)

// All ones where bit BIT of w is set, else 0 (one instruction; as C++ the and
// with it becomes an and, a compare and a select).
template <int BIT>
__device__ __forceinline__ int lane_mask(unsigned w) {
    int r;
    asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(r) : "v"(w), "n"(BIT));
    return r;
}

// Switches of the bonded terms (setSwitches_multi, MMFFmulti_lib.cpp:316-329).
struct FFSwitch {
    int doBonds, doPiPiI, doPiSigma, doAngles;
};

// -------------------------------------------------------------------------
// Bond stretch, Forces.h:137-143 (evalBond): f = h*(dl*k), E = k dl^2 / 2.
// pi-pi alignment, Forces.h:230-241 (evalPiAling) with ir1=ir2=1.
__device__ __forceinline__ float pi_align(V3 h1, V3 h2, float K, V3& f1, V3& f2) {
    float c = dot(h1, h2);
    f1 = h2 - h1 * c;
    f2 = h1 - h2 * c;
    bool sgn = c < 0.f;
    if (sgn) c = -c;
    float E = K * (1.f - c);
    float fang = sgn ? -K : K;
    f1 = f1 * fang;
    f2 = f2 * fang;
    return E;
}
// pi-sigma orthogonality, Forces.h:218-228 (evalAngleCos).
__device__ __forceinline__ float angle_cos(V3 h1, V3 h2, float ir1, float ir2, float K, float c0, V3& f1, V3& f2) {
    float c = dot(h1, h2);
    f1 = h2 - h1 * c;
    f2 = h1 - h2 * c;
    float c_ = c - c0;
    float E = K * c_ * c_;
    float fang = -K * c_ * 2.f;
    f1 = f1 * (fang * ir1);
    f2 = f2 * (fang * ir2);
    return E;
}
// sigma-sigma angle in the cos(theta/2) form, Forces.h:190-216
// (evalAngleCosHalf); cs0 = (cos(a0/2), sin(a0/2)).
__device__ __forceinline__ float angle_cos_half(V3 h1, V3 h2, float ir1, float ir2, float cs0x, float cs0y, float k,
                                                V3& f1, V3& f2) {
    V3 h = h1 + h2;
    float c2 = dot(h, h) * 0.25f;
    float s2 = 1.f - c2 + 1e-14f;
    float c = sqrtf(c2);
    float s = sqrtf(s2);
    // cs = cs0 udiv (c,s)  (Vec2.h:130)
    float csx = cs0x * c + cs0y * s;
    float csy = cs0y * c - cs0x * s;
    // k*(1 - csx) written as k*csy^2/(1 + csx) (|cs| = 1): no cancellation
    // near the equilibrium angle, where FP32 1 - csx loses the energy
    float E = k * csy * csy / (1.f + csx);
    float fr = -k * csy;
    c2 *= -2.f;
    fr /= 4.f * c * s;
    float fr1 = fr * ir1;
    float fr2 = fr * ir2;
    f1 = h * fr1 + h1 * (fr1 * c2);
    f2 = h * fr2 + h2 * (fr2 * c2);
    return E;
}

// -------------------------------------------------------------------------
// Bonded forces of one node, MMFFsp3_loc::eval_atom (MMFFsp3_loc.h:250-575)
// in the bNonBondNeighs strategy (bSubtractBondNonBond=false, ForceField.h:
// 168-184).  The 1-3 non-bonded subtraction of that function is not done
// here: the non-bonded sum excludes those pairs directly (see
// make_exclusions), which gives the same total force and energy.
// Outputs: recoils on the 4 neighbours (fbs) and on their pi-vectors (fps),
// the node's own force (fa) and its pi force (fpi).  Returns the energy.
// `pos(i)` returns the position of vec i (atom or, for i>=natoms, pi-vector);
// `nshift(k)` the periodic image shift of neighbour slot k (pbc_shifts of its
// neighCell, MMFFsp3_loc.h:325-329; zero in vacuum).
template <class PosFn, class ShiftFn>
__device__ __forceinline__ float eval_node(int ia, int natoms, int nnode, PosFn pos, ShiftFn nshift, const int4 ng,
                                           const float4 apar, const float4 bL, const float4 bK, const float4 ksp,
                                           const float4 kpp, const FFSwitch sw, V3* fbs, V3* fps, V3& fa, V3& fpi) {
    const V3 pa = pos(ia);
    const V3 hpi = pos(natoms + ia);
    const int ings[4] = {ng.x, ng.y, ng.z, ng.w};
    const float bLs[4] = {bL.x, bL.y, bL.z, bL.w};
    const float bKs[4] = {bK.x, bK.y, bK.z, bK.w};
    const float Ksp[4] = {ksp.x, ksp.y, ksp.z, ksp.w};
    const float Kpp[4] = {kpp.x, kpp.y, kpp.z, kpp.w};
    const float piC0 = apar.w;
    float E = 0.f;
    fa = zero3();
    fpi = zero3();
    V3 hs[4];
    float ir[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        fbs[i] = zero3();
        fps[i] = zero3();
    }
    int nb = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int ing = ings[i];
        if (ing < 0) break;
        nb = i + 1;
        V3 h = pos(ing) + nshift(i) - pa;
        const float l = sqrtf(dot(h, h));
        const float il = 1.f / l;
        h = h * il;
        hs[i] = h;
        ir[i] = il;
        V3 f1, f2;
        if (ia < ing) {
            if (sw.doBonds) {
                const float dl = l - bLs[i];
                const float fr = dl * bKs[i];
                f1 = h * fr;
                E += fr * dl * 0.5f;
                fbs[i] -= f1;
                fa += f1;
            }
            const float k = Kpp[i];
            if (sw.doPiPiI && (ing < nnode) && (k > 1e-6f)) {
                E += pi_align(hpi, pos(natoms + ing), k, f1, f2);
                fpi += f1;
                fps[i] += f2;
            }
        }
        const float k = Ksp[i];
        if (sw.doPiSigma && (k > 1e-6f)) {
            E += angle_cos(hpi, h, 1.f, il, k, piC0, f1, f2);
            fpi += f1;
            fa -= f2;
            fbs[i] += f2;
        }
    }
    if (sw.doAngles) {
        const float ssK = apar.z;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            if (i + 1 >= nb) break;
#pragma unroll
            for (int j = i + 1; j < 4; j++) {
                if (j >= nb) break;
                V3 f1, f2;
                E += angle_cos_half(hs[i], hs[j], ir[i], ir[j], apar.x, apar.y, ssK, f1, f2);
                fa -= f1 + f2;
                fbs[i] += f1;
                fbs[j] += f2;
            }
        }
    }
    return E;
}
// Vacuum molecules: no image shifts.
template <class PosFn>
__device__ __forceinline__ float eval_node(int ia, int natoms, int nnode, PosFn pos, const int4 ng, const float4 apar,
                                           const float4 bL, const float4 bK, const float4 ksp, const float4 kpp,
                                           const FFSwitch sw, V3* fbs, V3* fps, V3& fa, V3& fpi) {
    return eval_node(ia, natoms, nnode, pos, [](int) { return zero3(); }, ng, apar, bL, bK, ksp, kpp, sw, fbs, fps, fa,
                     fpi);
}

// Forces of eval_node for a vacuum molecule in LDS (pi-vector of node k at
// pos(pi0 + k)), without branches and without the energy: the neighbours are read at
// once, the four neighbours' norms and then the angles two by two run side by side,
// where the branches of eval_node wait for each read, root and division in turn (5800
// cycles a step for a wave of nodes, a third of them issuing).  Terms that a node does
// not have are computed on a unit vector and weighted zero.  The roundings are those
// that the compiler gives eval_node, written out.  put_pi(i, f) takes the recoil on
// neighbour i's pi-vector.  With the window reads below spread over the step, a system of
// 251 atoms takes 24.0 us a step instead of 25.4 (constant gains), and 512 molecules on
// the grid are scanned in 4.73 ms instead of 5.3.
template <class PosFn, class PutPi>
__device__ __forceinline__ void node_forces(int ia, int pi0, int nnode, PosFn pos, const int4 ng, const float4 apar,
                                            const float4 bL, const float4 bK, const float4 ksp, const float4 kpp,
                                            const FFSwitch sw, PutPi put_pi, V3* fbs, V3& fa, V3& fpi) {
#pragma clang fp contract(off)
    auto madd = [](V3 a, float k, V3 c) {
        return mk(__builtin_fmaf(a.x, k, c.x), __builtin_fmaf(a.y, k, c.y), __builtin_fmaf(a.z, k, c.z));
    };
    // computed here and not put off until the end, which would keep all operands
    auto now = [](V3& a) { asm volatile("" : "+v"(a.x), "+v"(a.y), "+v"(a.z)); };
    auto dotp = [](V3 a, V3 b) { return __builtin_fmaf(a.z, b.z, __builtin_fmaf(a.x, b.x, a.y * b.y)); };
    const int ings[4] = {ng.x, ng.y, ng.z, ng.w};
    const float bLs[4] = {bL.x, bL.y, bL.z, bL.w};
    const float bKs[4] = {bK.x, bK.y, bK.z, bK.w};
    const float Ksp[4] = {ksp.x, ksp.y, ksp.z, ksp.w};
    const float Kpp[4] = {kpp.x, kpp.y, kpp.z, kpp.w};
    bool has[4];
    V3 hs[4];
    float l[4], ir[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        has[i] = (i == 0 || has[i - 1]) && ings[i] >= 0;
        hs[i] = pos(has[i] ? ings[i] : ia);
    }
    const V3 pa = pos(ia);
    const V3 hpi = pos(pi0 + ia);
    fa = zero3();
    fpi = zero3();
#pragma unroll
    for (int i = 0; i < 4; i++) {
        V3 h = mk(hs[i].x - pa.x, hs[i].y - pa.y, hs[i].z - pa.z);
        h = mk(has[i] ? h.x : 1.f, has[i] ? h.y : 0.f, has[i] ? h.z : 0.f);
        l[i] = sqrtf(dotp(h, h));
        ir[i] = 1.f / l[i];
        hs[i] = mk(h.x * ir[i], h.y * ir[i], h.z * ir[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const V3 h = hs[i];
        const bool first = has[i] && ia < ings[i];
        const bool pin = has[i] && ings[i] < nnode;
        const V3 hp = pos(pi0 + (pin ? ings[i] : ia));
        float fr = (l[i] - bLs[i]) * bKs[i];  // bond
        fr = (first && sw.doBonds) ? fr : 0.f;
        fbs[i] = madd(h, -fr, zero3());
        fa = madd(h, fr, fa);
        float c = dotp(hpi, hp);  // pi-pi
        float k = (first && pin && sw.doPiPiI && Kpp[i] > 1e-6f) ? Kpp[i] : 0.f;
        k = c < 0.f ? -k : k;
        fpi = madd(madd(hpi, -c, hp), k, fpi);
        put_pi(i, madd(madd(hp, -c, hpi), k, zero3()));
        c = dotp(hpi, h);  // pi-sigma
        k = (has[i] && sw.doPiSigma && Ksp[i] > 1e-6f) ? Ksp[i] : 0.f;
        const float t = (c - apar.w) * -k;
        const float fang = t + t;
        const V3 f2 = madd(h, -c, hpi);
        fpi = madd(madd(hpi, -c, h), fang, fpi);
        fa = madd(f2, -(fang * ir[i]), fa);
        fbs[i] = madd(f2, fang * ir[i], fbs[i]);
        now(fa);
        now(fpi);
        now(fbs[i]);
    }
#pragma unroll
    for (int p = 0; p < 6; p++) {
        const int i = p < 3 ? 0 : (p < 5 ? 1 : 2), j = p < 3 ? p + 1 : (p < 5 ? p - 1 : 3);
        const V3 h = hs[i] + hs[j];
        const float d = __builtin_fmaf(h.z, h.z, __builtin_fmaf(h.y, h.y, h.x * h.x));
        const float c2 = d * 0.25f;
        const float s2 = __builtin_fmaf(d, -0.25f, 1.f) + 1e-14f;
        const float c = sqrtf(c2);
        const float s = sqrtf(s2);
        const float csy = __builtin_fmaf(apar.y, c, -(apar.x * s));
        float fr = (csy * -apar.z) / ((4.f * c) * s);
        fr = (has[j] && sw.doAngles) ? fr : 0.f;
        const float fr1 = fr * ir[i], fr2 = fr * ir[j];
        const float a1 = -2.f * c2 * fr1, a2 = -2.f * c2 * fr2;
        const V3 f1 = madd(h, fr1, mk(hs[i].x * a1, hs[i].y * a1, hs[i].z * a1));
        const V3 f2 = madd(h, fr2, mk(hs[j].x * a2, hs[j].y * a2, hs[j].z * a2));
        fa -= f1 + f2;
        fbs[i] += f1;
        fbs[j] += f2;
        if (p & 1) now(fa);
    }
}

// -------------------------------------------------------------------------
// Directed non-bonded pair, Forces.h:341-360 (getLJQH): bare Coulomb, LJ and
// the H-bond correction; REQ mixing Forces.h:270 (_mixREQ).  d = pj - pi;
// returns the force on i and the (unhalved) pair energy.
struct Req {
    float R, E, kQ, H;  // R0, sqrt(E0), COULOMB_K*Q, H
};
// 1/r from one v_rsq_f32 (1 ulp); the H-bond term is compiled in only for
// batches that carry H-bond charges (HB=true).
// PRECISE adds one Newton step to 1/r (energy passes: the Coulomb sums cancel
// to a small fraction of their terms, so a biased 1-ulp 1/r shows up there).
__device__ __forceinline__ float rsq_nr(float x) {
    const float y = __builtin_amdgcn_rsqf(x);
    return y * (1.5f - 0.5f * x * y * y);
}
template <bool HB = true, bool PRECISE = false>
__device__ __forceinline__ void lj_pair(V3 d, float Rij, float Eij, float kQQ, float Hij, float& fr, float& e) {
    const float r2 = dot(d, d);
    const float ir = PRECISE ? rsq_nr(r2) : __builtin_amdgcn_rsqf(r2);
    const float ir2 = ir * ir;
    const float Eq = kQQ * ir;
    const float u2 = (Rij * Rij) * ir2;
    const float u6 = u2 * u2 * u2;
    const float vdW = u6 * Eij;
    if (HB) {
        const float H = u6 * u6 * ((Hij < 0.f) ? Hij * Eij : 0.f);
        e = Eq + (u6 - 2.f) * vdW + H;
        fr = (Eq + ((u6 - 1.f) * vdW + H) * 12.f) * ir2;  // force on i = d * (-fr)
    } else {
        e = Eq + (u6 - 2.f) * vdW;
        fr = (Eq + (u6 - 1.f) * vdW * 12.f) * ir2;
    }
}

// Force factor of lj_pair<HB> alone (force on i = d * -fr), every rounding
// written out.
template <bool HB>
__device__ __forceinline__ float lj_force(V3 d, float Rij, float Eij, float kQQ, float Hij) {
#pragma clang fp contract(off)
    const float r2 = __builtin_fmaf(d.z, d.z, __builtin_fmaf(d.x, d.x, d.y * d.y));
    const float ir = __builtin_amdgcn_rsqf(r2);
    const float ir2 = ir * ir;
    const float u2 = (Rij * Rij) * ir2;
    const float u4 = u2 * u2;
    const float u6 = u2 * u4;
    const float vdW = Eij * u6;
    const float t = __builtin_fmaf(u2, u4, -1.f);
    float s;
    if (HB) s = __builtin_fmaf(t, vdW, ((Hij < 0.f) ? Eij * Hij : 0.f) * (u6 * u6));
    else s = t * vdW;
    return __builtin_fmaf(kQQ, ir, s * 12.f) * ir2;
}

// -------------------------------------------------------------------------
// Cubic B-spline GridFF sample, GridFF::getForce_Bspline (GridFF.h:355-402)
// -> Bspline::fe3d_pbc_comb3 (Bspline.h:742-809), basis/dbasis (:253-276).
// x,y periodic; z index truncated toward zero and clamped to [3, nz-5] while
// tz keeps the unclamped index (Bspline.h:746-759).
struct GridDev {
    const float4* coefs;  // (nx,ny,nz) float4 (P, L, Q, 0), z fastest
    int nx, ny, nz;
    float p0x, p0y, p0z;
    float isx, isy, isz;  // 1/step
    float rnx, rny;       // 1/nx, 1/ny (relaxation kernel)
};

__device__ __forceinline__ void bs_basis(float u, float* b) {
    const float inv6 = 1.f / 6.f;
    const float u2 = u * u;
    const float t = 1.f - u;
    b[0] = inv6 * t * t * t;
    b[1] = inv6 * (3.f * u2 * (u - 2.f) + 4.f);
    b[2] = inv6 * (3.f * u * (1.f + u - u2) + 1.f);
    b[3] = inv6 * u2 * u;
}
__device__ __forceinline__ void bs_dbasis(float u, float* d) {
    const float u2 = u * u;
    const float t = 1.f - u;
    d[0] = -0.5f * t * t;
    d[1] = 0.5f * (3.f * u2 - 4.f * u);
    d[2] = 0.5f * (-3.f * u2 + 2.f * u + 1.f);
    d[3] = 0.5f * u2;
}
__device__ __forceinline__ int imod(int i, int m) {
    int r = i % m;
    return r < 0 ? r + m : r;
}

// imod for the whole wave, rm = 1/m: below 2^22 the quotient from a float reciprocal is
// off by one at most (a third of the instructions of an integer division).
__device__ __forceinline__ int imod_near(int i, int m, float rm) {
    if (__any(i >= (1 << 22) || i <= -(1 << 22))) return imod(i, m);
    int r = i - (int)((float)i * rm) * m;
    r = r < 0 ? r + m : r;
    r = r < 0 ? r + m : r;
    return r >= m ? r - m : r;
}

// Returns E; adds the force to f.  plq = (cP, cL, cQ) of the atom.
__device__ __forceinline__ float grid_sample(const GridDev& g, V3 p, V3 plq, V3& f) {
    const float ux = (p.x - g.p0x) * g.isx;
    const float uy = (p.y - g.p0y) * g.isy;
    const float uz = (p.z - g.p0z) * g.isz;
    int ix = (int)ux, iy = (int)uy, iz = (int)uz;
    if (ux < 0.f) ix--;
    if (uy < 0.f) iy--;
    const float tx = ux - ix, ty = uy - iy, tz = uz - iz;
    iz = min(max(iz, 3), g.nz - 5);
    ix = imod(ix - 1, g.nx);
    iy = imod(iy - 1, g.ny);
    float bx[4], dx[4], by[4], dy[4], bz[4], dz[4];
    bs_basis(tx, bx);
    bs_dbasis(tx, dx);
    bs_basis(ty, by);
    bs_dbasis(ty, dy);
    bs_basis(tz, bz);
    bs_dbasis(tz, dz);
    float Fx = 0.f, Fy = 0.f, Fz = 0.f, E = 0.f;
#pragma unroll
    for (int a = 0; a < 4; a++) {
        int xa = ix + a;
        if (xa >= g.nx) xa -= g.nx;
        float ey = 0.f, fy = 0.f, fz = 0.f;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            int yb = iy + b;
            if (yb >= g.ny) yb -= g.ny;
            const float4* col = g.coefs + ((size_t)(xa * g.ny + yb) * g.nz + (iz - 1));
            float e = 0.f, de = 0.f;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float4 q = col[c];
                const float cs = plq.x * q.x + plq.y * q.y + plq.z * q.z;
                e += bz[c] * cs;
                de += dz[c] * cs;
            }
            fy += e * dy[b];
            fz += de * by[b];
            ey += e * by[b];
        }
        Fx += ey * dx[a];
        Fy += fy * bx[a];
        Fz += fz * bx[a];
        E += ey * bx[a];
    }
    f.x -= Fx * g.isx;
    f.y -= Fy * g.isy;
    f.z -= Fz * g.isz;
    return E;
}

// Basis values and derivatives of one axis for GridWave, every
// rounding written out (fused where __builtin_fmaf stands, nowhere else).
__device__ __forceinline__ void bs_weights(float u, float* b, float* d) {
#pragma clang fp contract(off)
    const float inv6 = 1.f / 6.f;
    const float u2 = u * u;
    const float t = 1.f - u;
    const float q = 3.f * u2;
    b[0] = t * (t * (inv6 * t));
    b[1] = inv6 * __builtin_fmaf(u - 2.f, q, 4.f);
    b[2] = inv6 * __builtin_fmaf(3.f * u, __builtin_fmaf(-u, u, u + 1.f), 1.f);
    b[3] = u * (inv6 * u2);
    d[0] = t * (-0.5f * t);
    d[1] = 0.5f * __builtin_fmaf(-4.f, u, q);
    d[2] = 0.5f * (__builtin_fmaf(2.f, u, -q) + 1.f);
    d[3] = 0.5f * u2;
}

// The same sample for the atoms of a whole wave (every lane calls; `act` marks
// the lanes with an atom, lane 0 among them) through a cache in global memory:
// each atom owns a slot of 16 float4 with the 4x4x4 window of channel-combined
// coefficients cs = plq . c, row r = a*4+b of the wave's n atoms at cache[r*n ..].
// The wave's slots are one run of 256 n bytes.  While an atom stays in the grid cell
// of its slot (window base `key`) the 64 gathers from the 10 MB grid become one read
// of the slot.
//
// A step moves a few of a wave's 64 atoms across a cell face (0.1 A), so nearly
// every step refills some slots.  A refill is done by the whole wave: lane l
// fetches coefficient (a, b, c) = (l>>4, (l>>2)&3, l&3) of the leaving atom's new
// window, one load instruction of 16 runs of 64 B, and stores its combined value
// into the slot.  Refilling in the atom's own lane instead takes 64 loads in a
// row with one or two lanes active, and was 60-80 % of the sample's time.
// Reads of the slots follow the stores of the same wave in program order.
//
// The calls are spread over the force phase so that no wave waits for memory:
// locate() starts the gathers of the first four leaving atoms before the bonded
// terms, refill() stores them after, and each half of the slot is read by fetch()
// before half of the pair loop and used by add() after it (a whole slot in flight
// would take 64 registers).
struct GridWave {
    V3 t = {};   // position in the cell
    int ix = 0, iy = 0, iz = 0;
    unsigned long long miss = 0;  // lanes whose slot holds another window
    int n0 = 0;  // gathers in flight from locate()
    float4 q0[4];
    float4 w[8];
    V3 F = {};   // sum over the window

    __device__ __forceinline__ GridWave() {
#pragma unroll
        for (int t = 0; t < 4; t++) any_value(q0[t]);
    }
    // starts the gathers of the first (up to B) atoms in `miss`; returns their number
    template <int B>
    __device__ __forceinline__ int gather(const GridDev& g, int lane, float4* q) {
        const int la = lane >> 4, lb = (lane >> 2) & 3, lc = (lane & 3) - 1;
        const int n = min((int)__popcll(miss), B);
        unsigned long long left = miss;
#pragma unroll
        for (int t = 0; t < B; t++) {
            any_value(q[t]);
            if (t >= n) continue;
            const int m = (int)__ffsll(left) - 1;
            left &= left - 1;
            int xa = __builtin_amdgcn_readlane(ix, m) + la;
            int yb = __builtin_amdgcn_readlane(iy, m) + lb;
            xa = min((unsigned)xa, (unsigned)(xa - g.nx));  // periodic: 0 <= xa < nx + 3
            yb = min((unsigned)yb, (unsigned)(yb - g.ny));
            q[t] = g.coefs[(size_t)(xa * g.ny + yb) * g.nz + (__builtin_amdgcn_readlane(iz, m) + lc)];
        }
        return n;
    }
    // stores the n gathered windows and takes their atoms out of `miss`
    template <int B>
    __device__ __forceinline__ void store(V3 plq, int lane, float4* cache, int stride, int n, const float4* q) {
#pragma clang fp contract(off)
        float* slot = reinterpret_cast<float*>(cache + (lane >> 2) * stride) + (lane & 3);
#pragma unroll
        for (int t = 0; t < B; t++) {
            if (t >= n) break;
            const int m = (int)__ffsll(miss) - 1;
            miss &= miss - 1;
            auto bcast = [&](float v) {
                return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), m));
            };
            const float cx = bcast(plq.x), cy = bcast(plq.y), cz = bcast(plq.z);
            slot[m * 4] = __builtin_fmaf(cz, q[t].z, __builtin_fmaf(cx, q[t].x, cy * q[t].y));
        }
    }
    __device__ __forceinline__ void locate(const GridDev& g, int lane, bool act, V3 p, int& key) {
#pragma clang fp contract(off)
        const float qx = p.x - g.p0x, qy = p.y - g.p0y, qz = p.z - g.p0z;
        const float ux = qx * g.isx, uy = qy * g.isy;
        ix = (int)ux;
        iy = (int)uy;
        iz = (int)(qz * g.isz);
        if (ux < 0.f) ix--;
        if (uy < 0.f) iy--;
        t = mk(__builtin_fmaf(g.isx, qx, -(float)ix), __builtin_fmaf(g.isy, qy, -(float)iy),
               __builtin_fmaf(g.isz, qz, -(float)iz));
        iz = min(max(iz, 3), g.nz - 5);
        ix = imod_near(ix - 1, g.nx, g.rnx);
        iy = imod_near(iy - 1, g.ny, g.rny);
        const int k = (ix * g.ny + iy) * g.nz + iz;
        miss = __ballot(act && k != key);
        key = act ? k : key;
        if (miss) n0 = gather<4>(g, lane, q0);
    }
    __device__ __forceinline__ void refill(const GridDev& g, int lane, V3 plq, float4* cache, int stride) {
        F = zero3();
        if (miss) {
            store<4>(plq, lane, cache, stride, n0, q0);
            while (miss) {
                float4 q[8];
                const int n = gather<8>(g, lane, q);
                store<8>(plq, lane, cache, stride, n, q);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
    __device__ __forceinline__ void fetch(int lane, const float4* cache, int stride, int half) {
        asm volatile("" : "+v"(lane));  // else the row addresses are kept over the pair loop
        const float4* mine = cache + half * 8 * stride + lane;
#pragma unroll
        for (int r = 0; r < 8; r++) w[r] = mine[r * stride];
    }
    __device__ __forceinline__ void no_fetch() {
#pragma unroll
        for (int r = 0; r < 8; r++) any_value(w[r]);
    }
    // adds the x-slabs 2*half and 2*half+1 of the window
    __device__ __forceinline__ void add(int half) {
#pragma clang fp contract(off)
        asm volatile("" : "+v"(t.x), "+v"(t.y), "+v"(t.z));  // else the 24 weights are kept over the pair loop
        float bx[4], dx[4], by[4], dy[4], bz[4], dz[4];
        bs_weights(t.x, bx, dx);
        bs_weights(t.y, by, dy);
        bs_weights(t.z, bz, dz);
#pragma unroll
        for (int a = 0; a < 2; a++) {
            float ey = 0.f, fy = 0.f, fz = 0.f;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const float4 cs = w[a * 4 + b];
                float e = __builtin_fmaf(bz[0], cs.x, 0.f), de = __builtin_fmaf(dz[0], cs.x, 0.f);
                e = __builtin_fmaf(bz[1], cs.y, e);
                de = __builtin_fmaf(dz[1], cs.y, de);
                e = __builtin_fmaf(bz[2], cs.z, e);
                de = __builtin_fmaf(dz[2], cs.z, de);
                e = __builtin_fmaf(bz[3], cs.w, e);
                de = __builtin_fmaf(dz[3], cs.w, de);
                fy = __builtin_fmaf(dy[b], e, fy);
                fz = __builtin_fmaf(by[b], de, fz);
                ey = __builtin_fmaf(by[b], e, ey);
            }
            const float b1 = half ? bx[a + 2] : bx[a], d1 = half ? dx[a + 2] : dx[a];
            F.x = __builtin_fmaf(ey, d1, F.x);
            F.y = __builtin_fmaf(fy, b1, F.y);
            F.z = __builtin_fmaf(fz, b1, F.z);
        }
    }
    __device__ __forceinline__ void finish(const GridDev& g, V3& f) const {
        f.x = __builtin_fmaf(-g.isx, F.x, f.x);
        f.y = __builtin_fmaf(-g.isy, F.y, f.y);
        f.z = __builtin_fmaf(-g.isz, F.z, f.z);
    }
};

// -------------------------------------------------------------------------
// Positional restraint and bounding wall of one atom at p, the terms of the
// reference's update kernel (updateAtomsMMFFf4, relax_multi.cl:997-1009):
//   restraint (c.w > 0):  f += (c.xyz - p) * max(k.xyz, 0)
//   wall on axis d with stiffness bc_d > 0:  f_d += (lo_d - p_d) bc_d below
//   lo_d, (hi_d - p_d) bc_d above hi_d  (the reference enables z only; x and
//   y follow the same rule when their stiffness is positive).
__device__ __forceinline__ V3 restraint_force(V3 p, float4 c, float4 k) {
    if (!(c.w > 0.f)) return zero3();
    return mk((c.x - p.x) * fmaxf(k.x, 0.f), (c.y - p.y) * fmaxf(k.y, 0.f), (c.z - p.z) * fmaxf(k.z, 0.f));
}
__device__ __forceinline__ float wall1(float x, float lo, float hi, float k) {
    if (!(k > 0.f)) return 0.f;
    return (x < lo) ? (lo - x) * k : ((x > hi) ? (hi - x) * k : 0.f);
}
__device__ __forceinline__ V3 wall_force(V3 p, float4 lo, float4 hi, float4 k) {
    return mk(wall1(p.x, lo.x, hi.x, k.x), wall1(p.y, lo.y, hi.y, k.y), wall1(p.z, lo.z, hi.z, k.z));
}

// -------------------------------------------------------------------------
// FIRE parameters (DynamicOpt.h:47-95 defaults; set_opt, MMFFmulti_lib.cpp:141)
struct FireParams {
    float dt_max, dt_min, damp_max, finc, fdec, falpha, cv_kill;
    int minLastNeg;
};
// Per-system FIRE state.
struct FireState {
    float dt, damping;
    int lastNeg;
};
// DynamicOpt::FIRE_update_params (DynamicOpt.cpp:250-267) with
// damp_func_FIRE (:210-222).  Returns (cv, cf_eff) where the velocity update
// is v = cv*v + (dt + cf_eff)*f and cf_eff = renorm*cf as passed by
// MolWorld_sp3::run_no_omp (MolWorld_sp3.h:2426).
__device__ __forceinline__ void fire_update(const FireParams& P, FireState& S, float vf, float vv, float ff, float& cv,
                                            float& cfe) {
    const float f_len = sqrtf(ff);
    const float v_len = sqrtf(vv);
    const float cos_vf = vf / (f_len * v_len + 1e-32f);
    const float renorm = v_len / (f_len + 1e-32f);
    float cf;
    if (cos_vf < 0.f) {
        cv = P.cv_kill;
        cf = 0.f;
    } else {
        cv = 1.f - S.damping;
        cf = S.damping;
    }
    cf *= renorm;
    if (cos_vf < 0.f) {
        S.dt = fmaxf(S.dt * P.fdec, P.dt_min);
        S.lastNeg = 0;
        S.damping = P.damp_max;
    } else {
        if (S.lastNeg > P.minLastNeg) {
            S.dt = fminf(S.dt * P.finc, P.dt_max);
            S.damping = S.damping * P.falpha;
        }
        S.lastNeg++;
    }
    cfe = renorm * cf;
}

// -------------------------------------------------------------------------
// Langevin drive of the exploring phase (updateAtomsMMFFf4,
// relax_multi.cl:1160-1178): f += -gamma*v + xi*sqrt(2*kB*T*gamma/dt) on atoms
// (pi-vectors are not driven), with xi a unit-variance random number per
// component.  xi comes from a counter-based hash of (seed, system, vec, axis,
// step) -- murmur3's 32-bit finaliser applied after each field -- mapped to a
// uniform on [-sqrt(3), sqrt(3)); integer arithmetic only, so the FP64 oracle
// draws the same numbers.
constexpr float BOLTZMANN_K = 8.617333262145e-5f;  // eV/K (cpp/common/constants.h:12)
__host__ __device__ inline unsigned fmix32(unsigned h) {
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    h *= 0xC2B2AE35u;
    h ^= h >> 16;
    return h;
}
__host__ __device__ inline unsigned drive_hash(unsigned seed, unsigned sys, unsigned vec, unsigned axis,
                                               unsigned step) {
    unsigned h = fmix32(seed + 0x9E3779B9u);
    h = fmix32(h ^ sys);
    h = fmix32(h ^ (vec * 3u + axis));
    return fmix32(h ^ step);
}
__device__ __forceinline__ float drive_xi(unsigned seed, unsigned sys, unsigned vec, unsigned axis, unsigned step) {
    const unsigned h = drive_hash(seed, sys, vec, axis, step) >> 8;  // 24 bits
    return ((float)h * (2.f / 16777216.f) - 1.f) * 1.7320508f;
}

}  // namespace fcd
