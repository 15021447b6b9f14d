// Persistent batched FIRE relaxation on gfx950.
//
// One workgroup relaxes one system at a time, entirely on the device: it
// pulls a system index from a global work queue (systems pre-sorted by
// decreasing cost, so the largest start first), stages the system in LDS,
// iterates force evaluation + per-system FIRE until the system's own Fmax is
// below tolerance (or it hits the step limit / goes non-finite), writes the
// result back and pulls the next system.  Retirement is therefore per system
// with no host round trip and no grid-wide barrier.
//
// Per FIRE step (reference recipe MolWorld_sp3::run_no_omp,
// MolWorld_sp3.h:2291-2474):
//   A. forces: thread i -> non-bonded pairs (i, i+k mod N), k <= N/2, with the
//      reactions in per-wave LDS rows (positions/params from LDS, exclusions
//      from an LDS bit matrix) + B-spline GridFF sample through the atom's
//      window cache; thread k -> bonded terms of node k (recoils into LDS,
//      MMFFsp3_loc.h:250-575)
//   B. assemble: thread v -> own force + reactions + recoils via
//      back-neighbours, pi force projected perpendicular to the pi-vector
//      (assemble_atom, :998-1021); optional rigid-body preconditioner
//      (precond.h); block reduction of <v|f>, <v|v>, <f|f> and max|f|^2
//   C. per-system FIRE (DynamicOpt.cpp:250-267) and move (move_atom_FIRE,
//      MMFFsp3_loc.h:1264-1281)
// The learned form pauses the step loop every P steps to evaluate the
// proposal network (proposal.h) and restarts that step with the new gains.
#include "kernels.h"
#include "precond.h"
#include "proposal.h"

namespace fcd {

// Four small signed indices (atoms, or recoil rows: below 2048) in two registers.
__device__ __forceinline__ uint2 pack4(int4 a) {
    return make_uint2(((unsigned)a.x & 0xFFFFu) | ((unsigned)a.y << 16), ((unsigned)a.z & 0xFFFFu) | ((unsigned)a.w << 16));
}
__device__ __forceinline__ int4 unpack4(uint2 p) {
    return make_int4((int)(short)p.x, (int)p.x >> 16, (int)(short)p.y, (int)p.y >> 16);
}

// LDS layout (bytes), computed identically on the host (world.cpp).
//   pos   float4[prow]          (x, y, z, Q) of the atoms as periodic rows: row r
//                              holds atom r mod N, so the partners of an atom at
//                              offsets 0..N/2 follow it without a wrap
//   pi    float4[mmax]          pi-vectors
//   fnb   float4[nmax]          bonded self force of node i; with gains (precond.h) the
//                              exact force of atom i afterwards
//   re    float2[prow]          (R0, sqrt(E0)) in the rows of pos
//   hb    float[prow]           H in the same rows (batches with H-bond charges)
//   facc  float4[nwave*frow]    per-wave reaction forces of the half-ring schedule:
//                              entry e of wave w's row is the reaction on atom
//                              (64w+e) mod N
//   fself float4[mmax]          bonded self forces of the pi-vectors
//   fng   float4[8*mmax]        recoils (sigma rows, then pi rows)
//   mask  uint[wmax*nmax]       rotated exclusion rows, [word][atom]: the whole words
//                              below the one of the last offset, which each
//                              thread keeps in a register
//   learned gains only:
//   h     bf16 rows            network activations (one of the two buffers), over
//                              re..mask, which the next step needs again or rewrites
//   nb    short4[nmax]          bonded neighbours during the network evaluation, after h
//   gain  float[mmax+PC_MAXC]   gains of the stars and the components, after all of these
//
// The step is bound by how many waves a CU holds, and LDS is given out in units of
// 1280 B: a form that exceeds 53760 B at 256 atoms, static part included, runs two
// workgroups there instead of three.  Rows that only their own thread reads are not kept
// twice, which pays for the periodic rows: no size and form needs more than with plain
// rows and wrapped indices, and 256 atoms with up to 128 nodes run three workgroups in
// every form; 768 of them with H-bond charges and constant gains take 45 us a step, with
// two workgroups per CU 54.
struct LdsLayout {
    int nmax, mmax, nwave, learned, h2lds, hb;
    __host__ __device__ static int r16(int b) { return (b + 15) & ~15; }
    // rows of the pairs the loop computes: offsets 0..N/2 rounded up to whole iterations.
    // The rows it reads ahead in the last iteration, and does not use, are two more: they
    // lie in the next array.
    __host__ __device__ static int prow_of(int n) { return n + (n >> 1) + 3; }
    __host__ __device__ int prow() const { return prow_of(nmax); }
    __host__ __device__ int wmax() const { return nmax >> 6; }
    __host__ __device__ int off_pos() const { return 0; }
    __host__ __device__ int off_pi() const { return off_pos() + prow() * 16; }
    __host__ __device__ int off_fnb() const { return off_pi() + mmax * 16; }
    __host__ __device__ int off_re() const { return off_fnb() + nmax * 16; }
    __host__ __device__ int off_hb() const { return off_re() + r16(prow() * 8); }
    __host__ __device__ int off_facc() const { return off_hb() + (hb ? r16(prow() * 4) : 0); }
    // entries of a wave's reaction row: lane l's partner at offset k lands at l+k
    __host__ __device__ int frow() const { return 64 + (nmax >> 1); }
    __host__ __device__ int off_fself() const { return off_facc() + nwave * frow() * 16; }
    __host__ __device__ int off_fng() const { return off_fself() + mmax * 16; }
    __host__ __device__ int off_mask() const { return off_fng() + 8 * mmax * 16; }
    __host__ __device__ int end_base() const { return off_mask() + nmax * wmax() * 4; }
    __host__ __device__ int hbytes() const { return r16(nmax * MLP_HS * 2); }
    __host__ __device__ int off_h() const { return off_re(); }
    __host__ __device__ int off_nb() const { return off_h() + hbytes(); }
    __host__ __device__ int off_gain() const {
        const int e = end_base(), n = off_nb() + nmax * 8;
        return r16((learned && n > e) ? n : e);
    }
    // the second activation buffer, where it is kept in LDS
    __host__ __device__ int off_h2() const { return off_gain() + r16((mmax + PC_MAXC) * 4); }
    __host__ __device__ int bytes() const {
        if (!learned) return end_base();
        return off_h2() + (h2lds ? hbytes() : 0);
    }
};

// Work queues: class c owns order[qoff[c] .. qoff[c]+qcnt[c]) and counter
// queue[c].  A workgroup of class `cls` drains its own queue, then steals from
// the queues of the smaller classes (its LDS layout and width fit them), so no
// launch idles while another still has systems.
struct Queues {
    const int* order;
    int qoff[4];
    int qcnt[4];
    int* counter;
    int lowest;  // smallest class index a workgroup may steal from (its own index: no stealing)
    unsigned short* hslot;  // learned gains: global activation rows, one slot per workgroup of this launch
};

// minimum resident waves per SIMD the register allocation must allow
constexpr int WAVES_PER_SIMD = 3;
template <int BLOCK, bool HB, int PC>
__global__ void __launch_bounds__(BLOCK, WAVES_PER_SIMD)
relax_persistent_kernel(BatchDev B, RunParams P, Queues Q, int cls,
                                                                 LdsLayout L) {
    extern __shared__ float4 lds_dyn[];
    char* lds = reinterpret_cast<char*>(lds_dyn);
    float4* s_pos = reinterpret_cast<float4*>(lds + L.off_pos());
    float4* s_pi = reinterpret_cast<float4*>(lds + L.off_pi());
    float2* s_re = reinterpret_cast<float2*>(lds + L.off_re());
    float* s_hb = reinterpret_cast<float*>(lds + L.off_hb());
    float4* s_fnb = reinterpret_cast<float4*>(lds + L.off_fnb());
    float4* s_fself = reinterpret_cast<float4*>(lds + L.off_fself());
    float4* s_fng = reinterpret_cast<float4*>(lds + L.off_fng());
    unsigned* s_mask = reinterpret_cast<unsigned*>(lds + L.off_mask());
    float4* s_facc = reinterpret_cast<float4*>(lds + L.off_facc());
    float* s_gain = reinterpret_cast<float*>(lds + L.off_gain());
    // activation buffers of the in-kernel network: LDS where the layout allows,
    // else the two halves of this workgroup's global slot
    unsigned short* s_h = reinterpret_cast<unsigned short*>(lds + L.off_h());
    unsigned short* g_h = L.h2lds ? reinterpret_cast<unsigned short*>(lds + L.off_h2())
                                  : (Q.hslot ? Q.hslot + (size_t)blockIdx.x * (L.hbytes() / 2) : nullptr);
    const bool learned = PC >= 2 && L.learned && P.pc_mode == 2;
    const bool inkernel = learned && P.chunk == 0;  // network evaluated inside this kernel
    constexpr int NW = BLOCK / 64;
    __shared__ float s_red[4][2 * NW];
    __shared__ double s_redd[NW];
    __shared__ int s_q;
    // preconditioner: per-wave partial sums and the fit of each component
    __shared__ float s_cred[PC ? NW : 1][PC ? PC_MAXC : 1][PC_NSUM];
    __shared__ float s_csum[PC ? PC_MAXC : 1][PC_NFIT];
    __shared__ float s_smax[NW];
    __shared__ float s_st_best;       // FIRE fallback of the learned form (below)
    __shared__ int s_st_cnt, s_st_plain;

    int cc = cls;
    for (;;) {
        const int tid = opaque_tid();
        if (tid == 0) {
            int q = -1;
            while (cc >= Q.lowest) {
                const int k = atomicAdd(Q.counter + cc, 1);
                if (k < Q.qcnt[cc]) {
                    q = Q.order[Q.qoff[cc] + k];
                    if (P.chunk > 0 && B.status[q] != ST_RUNNING) continue;  // finished in an earlier chunk
                    break;
                }
                cc--;
            }
            s_q = q;
        }
        __syncthreads();
        const int q = s_q;
        __syncthreads();
        if (q < 0) break;
        const int s = q;
        if (B.systime && tid == 0 && P.chunk == 0) B.systime[2 * s] = (long long)wall_clock64();
        const SysInfo I = B.info[s];
        const int N = I.natoms, M = I.nnode, V = N + M;
        const int sflags = B.sysflags ? B.sysflags[s] : 0;  // restraints (bit 0), walls (bit 1)
        const int W = (N + 31) >> 5;   // exclusion words per atom in memory
        // last offset of the half ring; without non-bonded terms 0, which leaves one masked
        // iteration of the pair loop, for the grid window's halves, and none in vacuum: all
        // offsets masked took 68 us a step for 4096 vacuum systems of 16..256 atoms, this 22
        const int Kl = P.bNonBonded ? N >> 1 : 0;
        const int Wh = Kl >> 5;        // its exclusion word, kept in a register; the words below it are in LDS
        const int PR = LdsLayout::prow_of(N);  // periodic rows of this system
        // exclusion rows transposed to [word][atom] so that lanes read consecutive banks
        auto stage_mask = [&] {
            for (int w = opaque_tid(); w < N * Wh; w += BLOCK) {
                const int a = w / Wh, wd = w - a * Wh;
                s_mask[wd * N + a] = B.excl_rot[I.mask0 + a * W + wd];
            }
        };
        auto stage_re = [&] {
            for (int r = opaque_tid(); r < PR; r += BLOCK) {
                const float4 q = B.REQs[I.a0 + r % N];
                s_re[r] = make_float2(q.x, q.y);
                if (HB) s_hb[r] = q.w;
            }
        };
        // row of vec v in s_pos, and the parameters of atom j as they were given
        auto vrow = [&](int v) { return v < N ? v : L.prow() + v - N; };
        auto req = [&](int j) {
            const float2 q = s_re[j];
            return make_float4(q.x, q.y, s_pos[j].w, HB ? s_hb[j] : 0.f);
        };

        // ---- stage the system in LDS
        for (int r = tid; r < PR; r += BLOCK) {
            const int a = r % N;
            const float4 p = B.atoms[I.v0 + a];
            s_pos[r] = make_float4(p.x, p.y, p.z, B.REQs[I.a0 + a].z);
        }
        for (int k = tid; k < M; k += BLOCK) s_pi[k] = B.atoms[I.v0 + N + k];
        stage_re();
        stage_mask();

        const int nc = PC ? B.ncomp[s] : 0;
        V3 vel[2];
#pragma unroll
        for (int r = 0; r < 2; r++) vel[r] = zero3();
        FireState fs;
        fs.dt = P.fire.dt_max;
        fs.damping = P.fire.damp_max;
        fs.lastNeg = 0;
        int step = 0;
        int gkey = -1;    // grid window held in this atom's cache slot (none yet)
        if (P.chunk > 0) {  // resume the suspended state of this system
            const float4 fst = B.fire[s];
            fs.dt = fst.x;
            fs.damping = fst.y;
            fs.lastNeg = (int)fst.z;
            step = B.nsteps[s];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int v = tid + r * BLOCK;
                if (v < V) vel[r] = xyz(B.avel[I.v0 + v]);
            }
        }
        // FIRE fallback of the learned form: the best block max|F|^2 seen at a
        // proposal point after step 0, the proposal points since it was last
        // improved, and whether the system has fallen back to plain FIRE (zero
        // gains, no more network evaluations) after P.pc_stall such points.
        // Chunks of the chunked form carry it in B.stall.
        // The state lives in LDS, written by thread 0 between barriers only.
        if (learned) {
            const bool resume = P.chunk > 0 && step > 0;
            const float4 t = resume ? B.stall[s] : make_float4(INFINITY, 0.f, 0.f, 0.f);
            if (tid == 0) {
                s_st_best = t.x;
                s_st_cnt = (int)t.y;
                s_st_plain = t.z != 0.f ? 1 : 0;
            }
            if (!inkernel) {  // chunked: gains from the network kernel between chunks
                const bool plain = t.z != 0.f;
                for (int k = tid; k < M; k += BLOCK) s_gain[k] = plain ? 0.f : B.gnode[I.n0 + k];
                if (tid < PC_MAXC) s_gain[M + tid] = plain ? 0.f : B.gcomp[s * PC_MAXC + tid];
            }
        }
        // called by every thread of the block with its own max|F|^2 at a proposal point
        auto stall_check = [&](float fm2t) {
            const int tid = opaque_tid();
            fm2t = wave_max(fm2t);
            if ((tid & 63) == 0) s_smax[tid >> 6] = fm2t;
            __syncthreads();
            if (tid == 0) {
                float m = s_smax[0];
                for (int w = 1; w < NW; w++) m = fmaxf(m, s_smax[w]);
                if (m < s_st_best) {
                    s_st_best = m;
                    s_st_cnt = 0;
                } else if (++s_st_cnt >= P.pc_stall) {
                    s_st_plain = 1;
                }
            }
            __syncthreads();
            if (s_st_plain)
                for (int k = tid; k < M + PC_MAXC; k += BLOCK) s_gain[k] = 0.f;
            __syncthreads();
        };
        const int step_end = (P.chunk > 0) ? step + P.chunk : 0x7fffffff;
        bool suspended = false;
        __syncthreads();

        int status = ST_RUNNING;
        V3 fv[2];
        // The learned form evaluates the network between segments of the step
        // loop (one segment per proposal period): the step loop breaks out at a
        // proposal step once its exact forces are assembled, the network runs
        // with the forces and velocities parked in memory, and the segment
        // resumes that step at the preconditioner.  Nothing of the step loop is
        // live across the network, so neither part adds to the other's registers.
        // gains of the current step proposed: resume it after its force assembly.
        // A chunk of the chunked learned form resumes the step it was suspended
        // at, whose exact forces it parked (the first chunk computes its own)
        bool fresh = learned && !inkernel && step > 0;
        for (;;) {
            bool propose_now = false;
            const int tid = opaque_tid();
            const bool hasAtom = tid < N;
            // ---- per-thread state of this segment: atom tid, node tid, vecs tid and tid+BLOCK
            // exclusion word of the half ring's last offset
            const unsigned mlast = hasAtom ? B.excl_rot[I.mask0 + tid * W + Wh] : 0u;
            const int myc = (PC && hasAtom) ? B.comp[I.a0 + tid] : 0;
            uint2 ngp = pack4(make_int4(-1, -1, -1, -1));
            if (tid < M) ngp = pack4(B.neighs[I.a0 + tid]);
            // parameters of atom and node tid, read again for every step (while the step before
            // reduces and moves): the pair loop and the preconditioner need the registers
            float4 apar, bL, bK, ksp, kpp;
            V3 plq;
            auto load_params = [&](int k) {
                const int n = max(I.n0 + min(k, M - 1), 0);  // some node's where there is none
                apar = B.apars[n];
                bL = B.bLs[n];
                bK = B.bKs[n];
                ksp = B.Ksp[n];
                kpp = B.Kpp[n];
                plq = xyz(B.PLQs[I.a0 + min(k, N - 1)]);
            };
            load_params(tid);
            uint2 bkp[2];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int v = tid + r * BLOCK;
                // back-neighbours as local indices into s_fng (sigma rows [0,4M), pi rows [4M,8M))
                int4 b = B.bkNeighs[I.v0 + min(v, V - 1)];
                if (v >= V) b = make_int4(-1, -1, -1, -1);
                const int base = I.n0 * 8;
                bkp[r] = pack4(make_int4(b.x >= 0 ? b.x - base : -1, b.y >= 0 ? b.y - base : -1,
                                         b.z >= 0 ? b.z - base : -1, b.w >= 0 ? b.w - base : -1));
            }
            for (;;) {
                const int tid = opaque_tid();
                asm volatile("" : "+v"(ngp.x), "+v"(ngp.y), "+v"(bkp[0].x), "+v"(bkp[0].y), "+v"(bkp[1].x), "+v"(bkp[1].y));
                const int lane = tid & 63;
                const int wid = tid >> 6;
                const bool hasAtom = tid < N;
                const bool hasNode = tid < M;
                if (B.snap && step % B.snap_every == 0 && step / B.snap_every < B.nsnap) {
                    float4* dst = B.snap + (size_t)(step / B.snap_every) * B.ntotV + I.v0;
                    for (int v = tid; v < V; v += BLOCK) {
                        const float4 p = s_pos[vrow(v)];
                        dst[v] = make_float4(p.x, p.y, p.z, 0.f);
                    }
                }
                float vf = 0.f, vv = 0.f, ff = 0.f, fm2 = 0.f;
                if (!fresh) {
                    // ================= A: forces (no energies inside the step loop)
                    // Half-ring pair schedule (Newton's third law): the thread of atom i
                    // takes the partners j = (i+k) mod N, k = 1..N/2, so every unordered
                    // pair is computed once.  The partners of a wave at offset k are the
                    // 64 consecutive atoms 64w+k .. 64w+63+k (mod N), a window that slides
                    // by one atom per offset.  The reaction on each partner is accumulated
                    // in registers and moves down one lane per offset with the window
                    // (DPP wave shift; the atom entering at lane 63 starts from zero); the
                    // reaction leaving at lane 0 is written to the wave's reaction row:
                    // entry k as it leaves, the last 64 by all lanes after the last
                    // offset.  Every entry is written once and read after the block
                    // barrier: no clearing, no atomics, no lane ordering.
                    //
                    // The loop is bound by VALU issue (4.6 cycles per instruction, three
                    // resident waves per SIMD), so everything but the pair itself is kept
                    // out of it.  Partners come from periodic rows at addresses that advance
                    // by a constant (no index wrap); the exclusion bit of an offset becomes
                    // a lane mask in one instruction and is applied in one; offsets are
                    // taken four per iteration, two computed side by side, with the rows of
                    // the next two on their way.  Offset 0 (an atom with itself) and the
                    // offsets past N/2 that round up the last iteration are masked as
                    // excluded pairs are.  31.5 instructions per offset; with wrapped
                    // indices and one offset at a time it took 40, and waited for LDS.
                    const int nwAct = (N + 63) >> 6;
                    const int nrow = 64 + Kl;       // entries of a wave's reaction row that hold a reaction
                    const int wu = __builtin_amdgcn_readfirstlane(wid);
                    V3 f = zero3();
                    // lanes without an atom carry the window only: their own atom sits far
                    // away with zero parameters, so each of their pair forces is exactly 0
                    const float4 p4 = s_pos[hasAtom ? tid : 0];
                    const V3 pi = hasAtom ? xyz(p4) : mk(1e4f, 1e4f, 1e4f);
                    float4 ri = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (hasAtom) ri = req(tid);
                    const float kQi = COULOMB_K * ri.z;
                    const bool onGrid = P.bGridFF && wu < nwAct;  // the atoms of a wave together
                    GridWave gw;
                    if (onGrid) gw.locate(P.grid, lane, hasAtom, pi, gkey);
                    if (hasNode) {
                        V3 fbs[4], fa, fpi;
                        auto pos = [&](int v) { return xyz(s_pos[v]); };
                        auto put = [&](int row, V3 g) { s_fng[row] = make_float4(g.x, g.y, g.z, 0.f); };
                        node_forces(tid, L.prow(), M, pos, unpack4(ngp), apar, bL, bK, ksp, kpp, P.sw,
                                    [&](int k, V3 g) { put(4 * M + tid * 4 + k, g); }, fbs, fa, fpi);
#pragma unroll
                        for (int k = 0; k < 4; k++) put(tid * 4 + k, fbs[k]);
                        s_fnb[tid] = make_float4(fa.x, fa.y, fa.z, 0.f);
                        s_fself[tid] = make_float4(fpi.x, fpi.y, fpi.z, 0.f);
                    }
                    float4* slots = B.gridcache + (size_t)(I.a0 + wu * 64) * 16;
                    const int nslot = min(64, N - wu * 64);
                    if (onGrid) gw.refill(P.grid, lane, plq, slots, nslot);
                    if (wu < nwAct && (Kl > 0 || onGrid)) {
                        const int ia = hasAtom ? tid : 0;
                        const float4* pp = s_pos + ia;
                        const float2* pr = s_re + ia;
                        const float* ph = s_hb + ia;
                        V3 acc = zero3();
                        struct Rows {
                            float4 p = {};
                            float2 r = {};
                            float h = 0.f;
                        };
                        auto rows = [&](int k) {
                            Rows q;
                            q.p = pp[k];
                            q.r = pr[k];
                            q.h = HB ? ph[k] : 0.f;
                            return q;
                        };
                        // address of the entry that leaves at the iteration's first offset
                        unsigned fout = (unsigned)(size_t)(
                            (__attribute__((address_space(3))) char*)(lds + L.off_facc() + wu * L.frow() * 16));
                        // the pair with the rows q: force on the partner = d * fr
                        auto pair = [&](const Rows& q, V3& d, float& fr) {
                            d = mk(q.p.x - pi.x, q.p.y - pi.y, q.p.z - pi.z);
                            fr = lj_force<HB>(d, ri.x + q.r.x, ri.y * q.r.y, kQi * q.p.w, ri.w * q.h);
                        };
                        // adds the pair, masked by bit `bit` of keep, and moves the window on
                        auto add = [&](V3 d, float fr, int keep) {
                            fr = __builtin_bit_cast(float, __builtin_bit_cast(int, fr) & keep);
                            f.x = __builtin_fmaf(-d.x, fr, f.x);
                            f.y = __builtin_fmaf(-d.y, fr, f.y);
                            f.z = __builtin_fmaf(-d.z, fr, f.z);
                            acc.x = __builtin_fmaf(d.x, fr, acc.x);
                            acc.y = __builtin_fmaf(d.y, fr, acc.y);
                            acc.z = __builtin_fmaf(d.z, fr, acc.z);
                        };
                        auto shift = [&] {
                            acc.x = dpp_shl1_zero(acc.x);
                            acc.y = dpp_shl1_zero(acc.y);
                            acc.z = dpp_shl1_zero(acc.z);
                        };
                        Rows a0, a1, b0, b1;
                        a0 = rows(0);
                        a1 = rows(1);
                        unsigned keep = 0;
                        const int Kn = (Kl & ~3) + 4;  // offsets taken: 0..Kn-1
                        const int kmid = (Kn >> 3) << 2;
                        if (onGrid) gw.fetch(hasAtom ? lane : 0, slots, nslot, 0);
                        else gw.no_fetch();
#pragma clang loop unroll(disable)
                        for (int k = 0;; k += 4) {
                            if (k == kmid && onGrid) {
                                gw.add(0);
                                gw.fetch(hasAtom ? lane : 0, slots, nslot, 1);
                            }
                            if ((k & 31) == 0) {  // the next exclusion word, as bits of the pairs to keep
                                const int w = k >> 5;
                                keep = ~(w < Wh ? s_mask[w * N + ia] : mlast);
                                if (w == 0) keep &= ~1u;
                                if (w == Wh) {  // nothing past N/2; for even N the pair at N/2 is the lower half's
                                    const int top = (Kl & 31) + ((!(N & 1) && tid >= Kl) ? 0 : 1);
                                    keep &= top < 32 ? (1u << top) - 1u : ~0u;
                                }
                            }
                            pp += 2;
                            pr += 2;
                            ph += 2;
                            b0 = rows(0);
                            b1 = rows(1);
                            V3 d0, d1;
                            float g0, g1;
                            pair(a0, d0, g0);
                            pair(a1, d1, g1);
                            add(d0, g0, lane_mask<0>(keep));
                            lane0_store(fout, 0, acc);
                            shift();
                            add(d1, g1, lane_mask<1>(keep));
                            lane0_store(fout, 16, acc);
                            shift();
                            pp += 2;
                            pr += 2;
                            ph += 2;
                            a0 = rows(0);
                            a1 = rows(1);
                            pair(b0, d0, g0);
                            pair(b1, d1, g1);
                            add(d0, g0, lane_mask<2>(keep));
                            lane0_store(fout, 32, acc);
                            shift();
                            add(d1, g1, lane_mask<3>(keep));
                            if (k + 4 == Kn) break;
                            lane0_store(fout, 48, acc);
                            shift();
                            keep >>= 4;
                            fout += 64;
                        }
                        if (onGrid) gw.add(1);
                        if (Kn - 1 + lane < nrow)
                            s_facc[wu * L.frow() + Kn - 1 + lane] = make_float4(acc.x, acc.y, acc.z, 0.f);
                    }
                    if (hasAtom) {
                        const int i = tid;
                        if (P.bNonBonded) {
                            // weighted corrections (ring topologies; empty for trees)
                            for (int c = 0; c < I.ncorr; c++) {
                                const PairCorrDev pc = B.corr[I.corr0 + c];
                                if (pc.i != i) continue;
                                const float4 pj = s_pos[pc.j];
                                const float4 rj = req(pc.j);
                                const V3 d = mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z);
                                float fr, ep;
                                lj_pair<HB>(d, ri.x + rj.x, ri.y * rj.y, kQi * rj.z, ri.w * rj.w, fr, ep);
                                f -= d * (fr * pc.w);
                            }
                        }
                    }
                    if (onGrid) gw.finish(P.grid, f);
                    const V3 fnb = f;  // non-bonded and grid force on atom tid
                    __syncthreads();

                    // ================= B: assemble + reductions
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        const int v = tid + r * BLOCK;
                        fv[r] = zero3();
                        if (v < V) {
                            V3 f = zero3();
                            const bool isPi = r > 0 || v >= N;  // N <= BLOCK
                            if (!isPi) {
                                f = fnb;
                                if (P.bNonBonded && N >= 2)
                                    for (int w = 0; w < nwAct; w++) {  // atom v: entries (v-64w) mod N + multiples of N
                                        int e = v - 64 * w;            // > -N: an active wave's first atom is below N
                                        e = (e < 0) ? e + N : e;
                                        const float4* row = s_facc + w * L.frow();
                                        for (; e < nrow; e += N) f += xyz(row[e]);
                                    }
                                if (v < M) f += xyz(s_fnb[v]);
                                if (sflags) {  // restraints and walls are part of the exact force
                                    const V3 p = xyz(s_pos[v]);
                                    if (sflags & 1) f += restraint_force(p, B.constr[I.a0 + v], B.constrK[I.a0 + v]);
                                    if (sflags & 2) f += wall_force(p, B.bbox[3 * s], B.bbox[3 * s + 1], B.bbox[3 * s + 2]);
                                }
                            } else {
                                f = xyz(s_fself[v - N]);
                            }
                            const int4 b = unpack4(bkp[r]);
                            const int b4[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
                            for (int k = 0; k < 4; k++) {
                                if (b4[k] < 0) break;
                                f += xyz(s_fng[b4[k]]);
                            }
                            if (isPi) {
                                const V3 p = xyz(s_pi[v - N]);
                                f -= p * dot(p, f);
                            }
                            fm2 = fmaxf(fm2, dot(f, f));  // convergence always on the exact force
                            fv[r] = f;
                        }
                    }
                } else {
                    // restart of a proposal step: its exact forces were parked before the network
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        const int v = tid + r * BLOCK;
                        fv[r] = zero3();
                        if (v < V) {
                            fv[r] = xyz(B.aforce[I.v0 + v]);
                            fm2 = fmaxf(fm2, dot(fv[r], fv[r]));
                        }
                    }
                }
                // a proposal point after step 0 (in-kernel: before the network runs;
                // chunked: at the start of a chunk, after the network kernel)
                if (learned && P.pc_stall > 0 && step > 0 && step % P.pc_every == 0 && (inkernel ? !fresh : fresh) &&
                    !s_st_plain)
                    stall_check(fm2);
                if (!fresh && step >= step_end) {
                    // chunk done: suspend with the exact forces of the current
                    // geometry (written back below), so that the network between
                    // chunks sees positions and forces of the same step
                    suspended = true;
                    break;
                }
                if (PC == 2 && inkernel && !fresh && step % P.pc_every == 0 && !s_st_plain) {  // uniform across the block
                    if (hasAtom) s_fnb[tid] = make_float4(fv[0].x, fv[0].y, fv[0].z, 0.f);
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        const int v = tid + r * BLOCK;
                        if (v < V) B.aforce[I.v0 + v] = make_float4(fv[r].x, fv[r].y, fv[r].z, 0.f);
                    }
                    propose_now = true;
                    break;
                }
                if (PC)
                    precondition<BLOCK>(P, s_pos, s_fnb, s_fself, s_fng, &s_cred[0][0][0], &s_csum[0][0], s_gain,
                                        learned, N, M, nc, myc, hasAtom, hasNode, unpack4(ngp), unpack4(bkp[0]), fv[0]);
                // FIRE sums: totals per chunk of 64 consecutive vecs (vec v = tid + r*BLOCK
                // lies in chunk wid + r*NW), added in chunk order, so that the result does
                // not depend on the workgroup width a system is relaxed with
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const int v = tid + r * BLOCK;
                    float pvf = 0.f, pvv = 0.f, pff = 0.f;
                    if (v < V) {
                        V3 f = fv[r];
                        const float f2 = dot(f, f);
                        if (P.Flimit > 0.f && f2 > P.Flimit * P.Flimit) f = f * (P.Flimit / sqrtf(f2));
                        fv[r] = f;
                        pvf = dot(vel[r], f);
                        pvv = dot(vel[r], vel[r]);
                        pff = dot(f, f);
                    }
                    const float t = wave_sum4(pvf, pvv, pff, 0.f);  // lane l: total of value l >> 4
                    if ((lane & 15) == 0 && lane < 48) s_red[lane >> 4][wid + r * NW] = t;
                }
                load_params(tid);  // for the energy of this geometry or the next step's bonded terms
                fm2 = wave_max(fm2);
                if (lane == 0) s_red[3][wid] = fm2;
                __syncthreads();
                vf = 0.f;
                vv = 0.f;
                ff = 0.f;
#pragma unroll
                for (int c = 0; c < 2 * NW; c++) {
                    vf += s_red[0][c];
                    vv += s_red[1][c];
                    ff += s_red[2][c];
                }
                fm2 = s_red[3][0];
#pragma unroll
                for (int w = 1; w < NW; w++) fm2 = fmaxf(fm2, s_red[3][w]);
                const float crit = (P.conv_mode == CONV_F2SUM) ? ff : fm2;
                if (!(ff == ff) || isinf(ff)) status = ST_NAN;
                else if (crit < P.Fconv2) status = ST_CONVERGED;
                else if (step >= P.nstep_max) status = ST_MAXSTEP;
                if (status != ST_RUNNING) {
                    // energy of this geometry: precise 1/r, FP64 accumulation and reduction
                    double epart = 0.0;
                    if (hasAtom && P.bNonBonded) {
                        const int i = tid;
                        const V3 pi = xyz(s_pos[i]);
                        const float4 ri = req(i);
                        const float kQi = COULOMB_K * ri.z;
                        double e = 0.0;  // each unordered pair once (half ring)
                        for (int k = 1; k <= Kl; k++) {
                            if (!(N & 1) && k == Kl && i >= Kl) break;
                            const unsigned mw = (k >> 5) < Wh ? s_mask[(k >> 5) * N + i] : mlast;
                            if ((mw >> (k & 31)) & 1u) continue;
                            const float4 pj = s_pos[i + k];
                            const float4 rj = req(i + k);
                            float fr, ep;
                            lj_pair<true, true>(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), ri.x + rj.x, ri.y * rj.y,
                                                kQi * rj.z, ri.w * rj.w, fr, ep);
                            e += (double)ep;
                        }
                        double ec = 0.0;  // directed corrections carry half of the pair energy each
                        for (int c = 0; c < I.ncorr; c++) {
                            const PairCorrDev pc = B.corr[I.corr0 + c];
                            if (pc.i != i) continue;
                            const float4 pj = s_pos[pc.j];
                            const float4 rj = req(pc.j);
                            float fr, ep;
                            lj_pair<true, true>(mk(pj.x - pi.x, pj.y - pi.y, pj.z - pi.z), ri.x + rj.x, ri.y * rj.y,
                                                kQi * rj.z, ri.w * rj.w, fr, ep);
                            ec += (double)ep * pc.w;
                        }
                        epart += e + 0.5 * ec;
                    }
                    if (hasAtom && P.bGridFF) {
                        V3 fd = zero3();
                        epart += (double)grid_sample(P.grid, xyz(s_pos[tid]), plq, fd);
                    }
                    if (hasNode) {
                        V3 fbs[4], fps[4], fa, fpi;
                        auto pos = [&](int v) { return xyz(s_pos[v]); };
                        epart += (double)eval_node(tid, L.prow(), M, pos, unpack4(ngp), apar, bL, bK, ksp, kpp, P.sw, fbs, fps, fa, fpi);
                    }
                    double ed = wave_sum_d(epart);
                    if (lane == 0) s_redd[wid] = ed;
                    __syncthreads();
                    if (tid == 0) {
                        double E = 0.0;
                        for (int w = 0; w < NW; w++) E += s_redd[w];
                        B.Esys[s] = E;
                        B.nsteps[s] = step;
                        B.status[s] = status;
                        B.Fmax[s] = sqrtf(fm2);
                    }
                    break;
                }

                // ================= C: FIRE + move
                float cv, cfe;
                fire_update(P.fire, fs, vf, vv, ff, cv, cfe);
                const float dt = fs.dt;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const int v = tid + r * BLOCK;
                    if (v < V) {
                        const bool isPi = v >= N;
                        V3 p = xyz(s_pos[vrow(v)]);
                        V3 f = fv[r];
                        if (isPi) f -= p * dot(p, f);
                        V3 w = vel[r] * cv + f * (dt + cfe);
                        if (isPi) w -= p * dot(p, w);
                        p += w * dt;
                        if (isPi) p = p * (1.f / sqrtf(dot(p, p)));
                        vel[r] = w;
                        if (isPi) {
                            s_pi[v - N] = make_float4(p.x, p.y, p.z, 0.f);
                        } else {
                            // the atom's periodic rows (a second one below N/2 + 3, a third
                            // only in molecules of less than 5 atoms); Q stays
                            const f32x3 t = {p.x, p.y, p.z};
                            *reinterpret_cast<f32x3*>(s_pos + v) = t;
                            for (int q = v + N; q < PR; q += N) *reinterpret_cast<f32x3*>(s_pos + q) = t;
                        }
                    }
                }
                step++;
                fresh = false;
                __syncthreads();
            }
            if (!propose_now) break;
            // ---- network evaluation between segments (learned form)
            {
            const int tid = opaque_tid();
            const bool hasAtom = tid < N;
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int v = tid + r * BLOCK;
                if (v < V) B.avel[I.v0 + v] = make_float4(vel[r].x, vel[r].y, vel[r].z, 0.f);
            }
            __syncthreads();
            propose_gains<BLOCK>(P, B.neighs + I.a0, B.elem + I.a0, s_pos, s_pi, s_fnb,
                                 reinterpret_cast<short4*>(lds + L.off_nb()), s_h, g_h, s_gain, &s_cred[0][0][0], N, M, nc, hasAtom ? B.comp[I.a0 + tid] : 0,
                                 hasAtom ? B.PLQs[I.a0 + tid] : make_float4(0, 0, 0, 0));
            stage_mask();  // the exclusion rows and the pair parameters were overwritten
            stage_re();    // by the activations
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int v = tid + r * BLOCK;
                if (v < V) vel[r] = xyz(B.avel[I.v0 + v]);
            }
            }
            fresh = true;
            __syncthreads();
        }
        {
        const int tid = opaque_tid();
        if (suspended && tid == 0) {
            B.fire[s] = make_float4(fs.dt, fs.damping, (float)fs.lastNeg, 0.f);
            B.nsteps[s] = step;
        }
        if (learned && tid == 0) B.stall[s] = make_float4(s_st_best, (float)s_st_cnt, s_st_plain ? 1.f : 0.f, 0.f);
        // ---- write back the final state of this system
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int v = tid + r * BLOCK;
            if (v < V) {
                if (step > 0) {  // else nothing has moved
                    const float4 p = s_pos[vrow(v)];
                    B.atoms[I.v0 + v] = make_float4(p.x, p.y, p.z, 0.f);
                }
                B.avel[I.v0 + v] = make_float4(vel[r].x, vel[r].y, vel[r].z, 0.f);
                // preconditioned forms keep the exact atom forces in s_fnb; a suspended
                // chunk holds them, assembled and not yet preconditioned, in fv
                const V3 fo = (PC && v < N && !suspended) ? xyz(s_fnb[v]) : fv[r];
                B.aforce[I.v0 + v] = make_float4(fo.x, fo.y, fo.z, 0.f);
            }
        }
        }
        if (B.systime && threadIdx.x == 0 && P.chunk == 0) B.systime[2 * s + 1] = (long long)wall_clock64();
        __syncthreads();
    }
}

#define FC_INST(BL, HB, PCF) \
    template __global__ void relax_persistent_kernel<BL, HB, PCF>(BatchDev, RunParams, Queues, int, LdsLayout);
#define FC_INST2(BL)      \
    FC_INST(BL, false, 0) \
    FC_INST(BL, true, 0)  \
    FC_INST(BL, false, 1) \
    FC_INST(BL, true, 1)  \
    FC_INST(BL, false, 2) \
    FC_INST(BL, true, 2)  \
    FC_INST(BL, false, 3) \
    FC_INST(BL, true, 3)
FC_INST2(64)
FC_INST2(128)
FC_INST2(192)
FC_INST2(256)
#undef FC_INST2
#undef FC_INST

template <bool HB, int PCF>
static const void* kernel_ptr(int block) {
    switch (block) {
        case 64: return (const void*)&relax_persistent_kernel<64, HB, PCF>;
        case 128: return (const void*)&relax_persistent_kernel<128, HB, PCF>;
        case 192: return (const void*)&relax_persistent_kernel<192, HB, PCF>;
        case 256: return (const void*)&relax_persistent_kernel<256, HB, PCF>;
        default: return nullptr;
    }
}
// pc: preconditioner mode 0 (off), 1 (constant gains), 2 (learned gains, network
// inside the kernel), 3 (learned gains read from memory: chunked execution)
static const void* kernel_ptr(int block, int hb, int pc) {
    switch (pc) {
        case 1: return hb ? kernel_ptr<true, 1>(block) : kernel_ptr<false, 1>(block);
        case 2: return hb ? kernel_ptr<true, 2>(block) : kernel_ptr<false, 2>(block);
        case 3: return hb ? kernel_ptr<true, 3>(block) : kernel_ptr<false, 3>(block);
        default: return hb ? kernel_ptr<true, 0>(block) : kernel_ptr<false, 0>(block);
    }
}

}  // namespace fcd

// Host launcher (C linkage inside the library).  qinfo = {off[4], cnt[4]}.
extern "C" hipError_t fc_launch_relax_persistent(int block, int hb, int ngroups, size_t lds_bytes, hipStream_t stream,
                                                 const fcd::BatchDev* B, const fcd::RunParams* P, const int* order,
                                                 const int* qinfo, int* counters, int cls, int nmax, int mmax,
                                                 int steal, unsigned short* hslot, int h2lds) {
    fcd::LdsLayout L{nmax, mmax, block / 64, P->pc_mode == 2 ? 1 : 0, h2lds, hb};
    fcd::Queues Q;
    Q.order = order;
    for (int c = 0; c < 4; c++) {
        Q.qoff[c] = qinfo[c];
        Q.qcnt[c] = qinfo[4 + c];
    }
    Q.counter = counters;
    Q.lowest = steal ? 0 : cls;
    Q.hslot = hslot;
    const void* k = fcd::kernel_ptr(block, hb, (P->pc_mode == 2 && P->chunk > 0) ? 3 : P->pc_mode);
    if (!k) return hipErrorInvalidValue;
    void* args[] = {(void*)B, (void*)P, (void*)&Q, (void*)&cls, (void*)&L};
    return hipLaunchKernel(k, dim3(ngroups), dim3(block), args, lds_bytes, stream);
}

// Scratch of the allocation-free relaxation (World::relax_noalloc): the queue
// counters, the queue order, the activation slots of the in-kernel network and
// the GridFF window cache of one relaxation, in one file-scope device array of
// FC_NOALLOC_SCRATCH_BYTES.  Each device holds its own copy at its own address
// until the process ends; host code uses the address returned here, never the
// array's name.
static __device__ __align__(256) unsigned char scratch[FC_NOALLOC_SCRATCH_BYTES];

// Device address of this device's scratch array (looked up once per device,
// with that device current).
extern "C" hipError_t fc_noalloc_scratch(void** ptr) {
    constexpr int kMaxDev = 64;
    static void* dev_ptr[kMaxDev] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDev) return hipErrorInvalidDevice;
    if (!dev_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        dev_ptr[dev] = p;
    }
    *ptr = dev_ptr[dev];
    return hipSuccess;
}

extern "C" int fc_relax_lds_bytes(int nmax, int mmax, int block, int learned, int h2lds, int hb) {
    fcd::LdsLayout L{nmax, mmax, block / 64, learned, h2lds, hb};
    return L.bytes();
}
// Where its arrays begin, in the order of the layout's list above, then the second
// activation buffer and the end.
extern "C" void fc_relax_lds_offsets(int nmax, int mmax, int block, int learned, int h2lds, int hb, int* out) {
    fcd::LdsLayout L{nmax, mmax, block / 64, learned, h2lds, hb};
    const int o[] = {L.off_pos(), L.off_pi(), L.off_fnb(), L.off_re(), L.off_hb(), L.off_facc(), L.off_fself(),
                     L.off_fng(), L.off_mask(), L.off_h(), L.off_nb(), L.off_gain(), L.off_h2(), L.bytes()};
    for (size_t k = 0; k < sizeof(o) / sizeof(o[0]); k++) out[k] = o[k];
}
// The same for a batch without H-bond charges (wmax, the exclusion words of an atom,
// follows from nmax).
extern "C" int fc_lds_bytes(int nmax, int mmax, int wmax, int block, int learned, int h2lds) {
    (void)wmax;
    return fc_relax_lds_bytes(nmax, mmax, block, learned, h2lds, 0);
}

// bf16 elements of one workgroup's global activation slot (the second buffer)
extern "C" int fc_hslot_elems(int nmax) {
    fcd::LdsLayout L{nmax, 1, 1, 1, 0, 0};
    return L.hbytes() / 2;
}

extern "C" hipError_t fc_persistent_occupancy(int block, int hb, int pc, size_t lds, int* nblocks) {
    const void* k = fcd::kernel_ptr(block, hb, pc);
    if (!k) return hipErrorInvalidValue;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(nblocks, k, block, lds);
}
