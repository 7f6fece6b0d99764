// gfx950 kernels of the CQBEM precompute (collocation path, inverse CQ
// transform, jump/B post-processing).
//
// Work decomposition (collocation, regular pairs): a block owns the columns of
// a patch of vertices for some rows i at one frequency l and evaluates every
// face that touches the patch once, one lane per face (k_colloc_gh_patch).  Each
// output block is written exactly once, with no atomics; x_i and the frequency
// constants live in scalar registers.  The star form (k_colloc_gh,
// CQBEM_COLLOC_KERNEL=star) has a lane per output block instead, which integrates
// the faces of its column vertex's star.  Faces touching i (the singular ones)
// are skipped and integrated by the singular kernels, which own rows (i, l) and
// add into them.
//
// Reference counterparts: compute_elastodynamic_{G,H,B_trans,B_angular}_kernel_collocation
// (src/elastodynamics_cqbem_*_collocation.cu) and the inverse transform loops
// of src/elastodynamics_cqbem_{G,H,B_trans,B_angular}.cu.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "cqbem_device.hpp"
#include "cqbem_kernels.hpp"

namespace cqbem {

__device__ inline bool same_vertex(const Geom &g, int a, int b) {
    return a == b || (g.vmap != nullptr && g.vmap[a] == g.vmap[b]);
}

// ------------------------------------------------------------------------
// G and H, regular (non-touching) faces.  Grid: (ceil(nv/64), nl, rows).
// ------------------------------------------------------------------------
template <bool DG, bool DH>
__global__ void __launch_bounds__(64) k_colloc_gh(Geom g, const double4 *__restrict__ quad, int npts,
                                                   const Freq *__restrict__ freqs, int l0, Mat m, int row0,
                                                   cd *__restrict__ UG, cd *__restrict__ UH, long long ld,
                                                   long long lstride) {
    const int j = blockIdx.x * 64 + threadIdx.x;
    const int il = blockIdx.z;
    const int i = row0 + il;
    const int l = blockIdx.y;
    if (j >= g.nv) return;
    const Freq f = freqs[l0 + l];
    const double x0 = g.V[3 * i], x1 = g.V[3 * i + 1], x2 = g.V[3 * i + 2];
    cd ga[6], gb = {0, 0}, hh[9];
    for (int k = 0; k < 6; k++) ga[k] = cd{0, 0};
    for (int k = 0; k < 9; k++) hh[k] = cd{0, 0};

    const int t_end = g.vs_ptr[j + 1];
    for (int t = g.vs_ptr[j]; t < t_end; ++t) {
        const int pk = g.vs_face[t];
        const int fc = pk >> 2, c = pk & 3;
        const int a0 = g.F[3 * fc], a1 = g.F[3 * fc + 1], a2 = g.F[3 * fc + 2];
        if (same_vertex(g, i, a0) || same_vertex(g, i, a1) || same_vertex(g, i, a2)) continue;
        const double *p0 = g.V + 3 * a0, *p1 = g.V + 3 * a1, *p2 = g.V + 3 * a2;
        const double y00 = p0[0], y01 = p0[1], y02 = p0[2];
        const double y10 = p1[0], y11 = p1[1], y12 = p1[2];
        const double y20 = p2[0], y21 = p2[1], y22 = p2[2];
        const double n0 = g.N[3 * fc], n1 = g.N[3 * fc + 1], n2 = g.N[3 * fc + 2];
        const double ar = g.area[fc];
        cd v1[3], v2[3], s2 = {0, 0}, m4[6];
        if (DH) {
            for (int k = 0; k < 3; k++) v1[k] = v2[k] = cd{0, 0};
            for (int k = 0; k < 6; k++) m4[k] = cd{0, 0};
        }
        for (int q = 0; q < npts; ++q) {
            const double4 Q = quad[q];
            const double r0 = Q.x * y00 + Q.y * y10 + Q.z * y20 - x0;
            const double r1 = Q.x * y01 + Q.y * y11 + Q.z * y21 - x1;
            const double r2 = Q.x * y02 + Q.y * y12 + Q.z * y22 - x2;
            const double d2 = r0 * r0 + r1 * r1 + r2 * r2;
            const double ir = rsqrt_nr(d2), r = d2 * ir, ir2 = ir * ir;
            const double h0 = r0 * ir, h1 = r1 * ir, h2 = r2 * ir;
            const double bc = c == 0 ? Q.x : (c == 1 ? Q.y : Q.z);
            const double wL = Q.w * ar * bc;
            const Expo E = expo(r, f);
            if (DG) {
                cd al, be;
                g_coef(E, ir, ir2, m, al, be);
                const double wr = wL * ir;
                al = al * wr;
                fma_cr(gb, be, wr);
                fma_cr(ga[0], al, h0 * h0);
                fma_cr(ga[1], al, h1 * h1);
                fma_cr(ga[2], al, h2 * h2);
                fma_cr(ga[3], al, h0 * h1);
                fma_cr(ga[4], al, h0 * h2);
                fma_cr(ga[5], al, h1 * h2);
            }
            if (DH) {
                cd c1, c2, c4;
                h_coef(E, ir, ir2, f, m, c1, c2, c4);
                const double rn = h0 * n0 + h1 * n1 + h2 * n2;
                c1 = c1 * wL;
                c2 = c2 * wL;
                c4 = c4 * (wL * rn);
                fma_cr(v1[0], c1, h0), fma_cr(v1[1], c1, h1), fma_cr(v1[2], c1, h2);
                fma_cr(v2[0], c2, h0), fma_cr(v2[1], c2, h1), fma_cr(v2[2], c2, h2);
                fma_cr(s2, c2, rn);
                fma_cr(m4[0], c4, h0 * h0);
                fma_cr(m4[1], c4, h1 * h1);
                fma_cr(m4[2], c4, h2 * h2);
                fma_cr(m4[3], c4, h0 * h1);
                fma_cr(m4[4], c4, h0 * h2);
                fma_cr(m4[5], c4, h1 * h2);
            }
        }
        if (DH) {
            const double n[3] = {n0, n1, n2};
            for (int a = 0; a < 3; a++)
                for (int b = 0; b < 3; b++) {
                    cd v = m4[sidx(a, b)];
                    fma_cr(v, v1[a], n[b]);
                    fma_cr(v, v2[b], n[a]);
                    if (a == b) v += s2;
                    hh[a * 3 + b] += v;
                }
        }
    }
    const long long base = (long long)l * lstride + (long long)(3 * il) * ld + 3 * (long long)j;
    for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++) {
            if (DG) {
                cd v = ga[sidx(a, b)];
                if (a == b) v += gb;
                UG[base + a * ld + b] = v;
            }
            if (DH) UH[base + a * ld + b] = hh[a * 3 + b] * kInv4Pi;
        }
}


// ------------------------------------------------------------------------
// G and H, regular faces, patch form.  Column vertices are grouped into
// compact patches of at most kPatchVerts vertices; a block owns one (patch,
// frequency, row vertex) and evaluates every face touching the patch once, one
// lane per face, 64 faces (a chunk) per wave.  The lane runs the rule in the
// face's own frame (FaceFrame, point_g, point_h), where G has 6 and H 8
// different entries, and keeps the sums of all three corner basis functions in
// registers (84 doubles with G and H); the rule's points and weights are
// wave-uniform (scalar loads).  After the rule it rotates each corner's sums to
// the global axes and adds them to per-vertex LDS accumulators.  The waves add in
// chunk order (an LDS turn counter) and, within a chunk, in sub-steps that the
// host schedules so that no vertex is updated twice in one sub-step: every sum
// has one order, whatever the hardware's.  The block then writes each (row,
// column) block once.  The first and the last frequency of an even L, where s is
// real, are one slot (T = rp: two real numbers in the place of a complex one).
//
// Bound by FP64 VALU issue (and, near full issue, by the clock that the power
// limit leaves): 268 VALU instructions per point, of which 84 are the corner
// sums and 49 the two complex exponentials (exp_pair), and 1100 per face and row
// outside the rule.  Icosphere level 4, L = 32, 28 points (6.2e9 unique
// evaluations): 72 ms; 77 at 296 instructions, with the exponentials through
// reductions and e^x, sin, cos, as frequencies beyond the table's reach still
// have them; 81 with a slot for each real frequency.  The form it replaces, two
// lanes per face that swapped every point's 16 global entries through DPP, took
// 128 ms at 516 instructions per point.  Tried and slower: the same with a
// block barrier per sub-step (86.5 ms), the rotation inside the wave's turn
// (84 ms: it serializes the block), LDS atomic adds instead of the turn's
// 16-byte read-modify-writes (84 ms).  FP64 matrix instructions share the
// vector FP64 unit here (a 4x4x4 one takes 16 cycles and does not overlap with
// vector FMAs), so corner sums on them would cost 4 slots where 3 FMAs do.
// ------------------------------------------------------------------------
constexpr int kPatchVerts = 256;    // vertex slots per patch (60 KB of LDS accumulators)
constexpr int kPatchThreads = 256;
constexpr int kPatchPairs = 15;     // complex words per slot: G (6, packed symmetric) then H (9)
constexpr int kRmw = 8;             // slot words read at a time when a corner is added
constexpr int kNoStep = 0xff;       // sub-step code of a corner outside the patch
constexpr int kFramePairs = 3;      // per lane, read at every point: the FaceFrame

// A pointer that every lane holds alike, in scalar registers.
template <class T> __device__ inline T *uniform_ptr(T *p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v), hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (T *)((unsigned long long)hi << 32 | lo);
}
// A pointer read from memory, known to be to global memory.
template <class T> __device__ inline T *as_global(T *p) { return (T *)(__attribute__((address_space(1))) T *)p; }

// Orders the LDS accesses of the lanes of a wave: what any lane wrote before it, every lane reads after it.  No instruction
// (a wave's LDS accesses complete in order); it holds the compiler, which otherwise orders one lane's accesses only.
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Waits until the LDS counter holds `v`.  Every wave of the block is resident and every wave's waits are for events that
// earlier program points of the others raise, so each wait ends.
__device__ inline void wait_for(int *counter, int v) {
    while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(counter, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP)) != v)
        __builtin_amdgcn_s_sleep(1);
}

// Whether one of the first N vertices t and one of the face's corners c are the same mesh vertex (same_vertex of every
// pair), without a branch per pair.
template <int N>
__device__ inline bool touches(const Geom &g, const int (&t)[3], const int (&c)[3]) {
    int tt[3] = {t[0], t[1], t[2]}, cc[3] = {c[0], c[1], c[2]};
    if (g.vmap) {
#pragma unroll
        for (int k = 0; k < 3; k++) tt[k] = g.vmap[t[k]], cc[k] = g.vmap[c[k]];
    }
    bool any = false;
#pragma unroll
    for (int k = 0; k < N; k++)
#pragma unroll
        for (int j = 0; j < 3; j++) any |= tt[k] == cc[j];
    return any;
}

// The rows il0 .. il0 + nr - 1 of one (patch pc, frequency l) for a block of kPatchThreads threads.  acc, frame,
// exps (the table of the exponentials) are the block's LDS; callers that run another tile on the same LDS synchronise
// first.  The block has no barrier between its rows: a wave evaluates its first chunk of the next row before it writes
// out (and clears) its 64 vertex slots of the last one, so neither the other waves' adds nor the stores are waited for.
// `dest` returns where the rows go (PatchDest); it is called at each write-out, so that a caller that reads it from memory
// need not hold it in registers.
struct PatchDest {
    const int *patch_verts;
    cd *UG, *UH;
    long long ld, lstride;
};
template <bool DG, bool DH, bool GAL, class F, class Dest>
__device__ __attribute__((always_inline)) inline void patch_tile(const Geom &g, const double4 *__restrict__ ref_pts, int ref_npts,
                                 const Bands &bands, const F &f, const Mat &m, int row0, const double4 *__restrict__ tpts,
                                 const int *__restrict__ patch_chunk, const int4 *__restrict__ chunk_info,
                                 const int4 *__restrict__ chunk_faces, const Dest &dest, int pc, int l,
                                 int il0, int nr, double2 *acc, double2 *frame, double2 *exps) {
    typedef typename F::value T;
    constexpr int kWaves = kPatchThreads / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int k = tid; k < kPatchPairs * kPatchVerts; k += kPatchThreads) acc[k] = make_double2(0.0, 0.0);
    fill_exp_table(f, exps);
    // chunks added so far; waves that cleared their slots, over all rows: in the table's unused place, so that
    // two blocks fill a CU's LDS exactly
    int *turns = reinterpret_cast<int *>(exps + kExpCounters), *cleared = turns + 1;
    if (tid < 2) turns[tid] = 0;
    __syncthreads();
    // With one or two chunks, 4 or 2 waves share a chunk, each taking every 4th or 2nd point of the rule, as long as 7
    // points of the reference rule are left to each (a far row may leave a wave none: part_has_points).
    const_int *pch = (const_int *)(patch_chunk + pc);
    const int c0 = pch[0], nchunk = pch[1] - c0;
    const int split = nchunk == 1 && ref_npts >= 28 ? 4 : nchunk <= 2 && ref_npts >= 14 ? 2 : 1;
    const int nturn = nchunk * split;

    // writes the G and H blocks of (row r of the tile, the wave's vertex slots) and clears the slots
    auto write_row = [&](int r) {
        wait_for(turns, (r + 1) * nturn);
        const PatchDest D = dest();
        const int j = D.patch_verts[pc * kPatchVerts + tid];
        if (j >= 0) {
            // cd: one complex entry at frequency l; rp: the real entries at frequencies 0 and l
            constexpr bool kReal = std::is_same<T, rp>::value;
            const long long obase = (kReal ? 0 : (long long)l * D.lstride) + (long long)(3 * (il0 + r)) * D.ld + 3 * (long long)j;
            auto put = [&](cd *o, const double2 &w, double scale) {
                *o = kReal ? cd{w.x * scale, 0.0} : cd{w.x * scale, w.y * scale};
                if (kReal) o[(long long)l * D.lstride] = cd{w.y * scale, 0.0};
            };
#pragma unroll
            for (int p = 0; p < 3; p++) {
#pragma unroll
                for (int b = 0; b < 3; b++) {
                    const int e = sidx(p, b);
                    if (DG) put(D.UG + obase + p * D.ld + b, acc[e * kPatchVerts + tid], m.g_scale);
                    if (DH) put(D.UH + obase + p * D.ld + b, acc[(6 + p * 3 + b) * kPatchVerts + tid], kInv4Pi);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int e = DG ? 0 : 6; e < (DH ? kPatchPairs : 6); e++) acc[e * kPatchVerts + tid] = make_double2(0.0, 0.0);
        wave_sync();  // every lane's words are cleared
        if (lane == 0) __hip_atomic_fetch_add(cleared, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    };

    // turn t of the tile: chunk part t % nturn of row t / nturn; the waves take the turns round robin over all rows, so
    // that a chunk count that is no multiple of the waves leaves none idle
    int written = 0;  // rows the wave has written out
#pragma unroll 1
    for (int t = wave; t < nr * nturn; t += kWaves) {
        const int r = t / nturn, turn = t - r * nturn, i = row0 + il0 + r;
        // the row point: vertex i (collocation), or test point i with its face's corners tv[] excluded (Galerkin)
        double x0, x1, x2;
        int tv[3] = {i, i, i};
        if (GAL) {
            const double4 P = tpts[i];
            x0 = P.x, x1 = P.y, x2 = P.z;
            const int f1 = (int)P.w;
            tv[0] = g.F[3 * f1], tv[1] = g.F[3 * f1 + 1], tv[2] = g.F[3 * f1 + 2];
        } else {
            x0 = g.V[3 * i], x1 = g.V[3 * i + 1], x2 = g.V[3 * i + 2];
        }
        const double4 *pts = ref_pts;
        int npts = ref_npts;
        if (bands.far_pts) {  // the row's rule: block-uniform (patch and row are)
            if (__builtin_amdgcn_readfirstlane((int)beyond_sphere(x0, x1, x2, bands.sphere[pc])))
                pts = bands.far_pts, npts = bands.far_npts;
        }
        pts = uniform_ptr(pts);
        const int part = turn % split;
        const_int *ci = as_const(chunk_info + (c0 + turn / split));
        const int4 info = make_int4(ci[0], ci[1], ci[2], 0);
        // lanes past the chunk's faces repeat its last one; they and the faces touching the row point are not added
        const int entry = info.x + min(lane, info.y - 1);
        const int4 fe = chunk_faces[entry];
        const int va[3] = {fe.x & 0xffffff, fe.y & 0xffffff, fe.z & 0xffffff};
        const bool touch = touches<GAL ? 3 : 1>(g, tv, va);
        const bool active = (lane < info.y) & !touch;
        const unsigned long long act = __builtin_amdgcn_ballot_w64(active);
        T sg[3][6], sh[3][8];
        if (act && part_has_points(npts, part)) {  // wave-uniform: no divergent merge of the sums
            {
                double y[3][3];
#pragma unroll
                for (int k = 0; k < 3; k++)
#pragma unroll
                    for (int d = 0; d < 3; d++) y[k][d] = g.V[3 * va[k] + d];
                const FaceFrame ff = face_frame(y, x0, x1, x2);
                frame[tid] = make_double2(ff.L1, ff.u), frame[kPatchThreads + tid] = make_double2(ff.v, ff.xa);
                frame[2 * kPatchThreads + tid] = make_double2(ff.xb, ff.cr);
            }
            // one point's entries into the sums; the first point starts them
            auto point = [&](int q, auto first) __attribute__((always_inline)) {
                // the lane is found anew at each point, so that neither the frame (12 VGPRs) nor the lane's number is held
                // through the loop
                unsigned all = ~0u;
                asm volatile("" : "+s"(all));
                const double2 *fr = frame + 64 * wave + __builtin_amdgcn_mbcnt_hi(all, __builtin_amdgcn_mbcnt_lo(all, 0));
                const double2 F0 = fr[0], F1 = fr[kPatchThreads], F2 = fr[2 * kPatchThreads];
                const_double *B = as_const(pts + 2 * q);  // b1, b2, -, -, w (phi_0, phi_1, phi_2, 1)
                const double ar = fma(B[0], F0.x, fma(B[1], F0.y, F1.y)), br = fma(B[1], F1.x, F2.x), cr = F2.y;
                const PointExpo<T> E = point_expo(fma(ar, ar, fma(br, br, cr * cr)), f, exps);
                const double w[3] = {B[4], B[5], B[6]};
                const double a = ar * E.ir, b = br * E.ir, c = cr * E.ir;
                auto add = [&](T &s, const T &v, double wk) {
                    if (first()) s = v * wk;
                    else fma_cr(s, v, wk);
                };
                // G and H one after the other, so that only one set of entries is live beside the sums
                __builtin_amdgcn_sched_barrier(0);
                if (DG) {
                    T G[6];
                    point_g(E, a, b, c, m, G);
#pragma unroll
                    for (int k = 0; k < 3; k++)
#pragma unroll
                        for (int e = 0; e < 6; e++) add(sg[k][e], G[e], w[k]);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (DH) {
                    T H[8];
                    point_h(E, a, b, c, m, H);
#pragma unroll
                    for (int k = 0; k < 3; k++)
#pragma unroll
                        for (int e = 0; e < 8; e++) add(sh[k][e], H[e], w[k]);
                }
            };
            each_part_point(npts, split, part, point);
        } else {
#pragma unroll
            for (int k = 0; k < 3; k++) {
#pragma unroll
                for (int e = 0; e < 6; e++) sg[k][e] = T{0, 0};
#pragma unroll
                for (int e = 0; e < 8; e++) sh[k][e] = T{0, 0};
            }
        }
        while (written < r) write_row(written++);
        // rotate each corner's sums and add them in the scheduled sub-steps, after every earlier chunk of the row and
        // once all slots are cleared
        const int4 ge = chunk_faces[info.x + min(lane, info.y - 1)];
        double Q[3][3], A[3][3];
        {
            double e1[3], e2[3], L1, area2;
            const int v0 = ge.x & 0xffffff, v1 = ge.y & 0xffffff, v2 = ge.z & 0xffffff;
            for (int d = 0; d < 3; d++) e1[d] = g.V[3 * v1 + d] - g.V[3 * v0 + d], e2[d] = g.V[3 * v2 + d] - g.V[3 * v0 + d];
            face_axes(e1, e2, Q, &L1, &area2);
            for (int j = 0; j < 3; j++)
                for (int k = 0; k < 3; k++) A[j][k] = Q[j][k] * (0.5 * area2);
        }
        double v[3][2 * kPatchPairs];
#pragma unroll
        for (int k = 0; k < 3; k++) {
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if (DG) {
                    double S[6], R[6];
#pragma unroll
                    for (int e = 0; e < 6; e++) S[e] = p ? sg[k][e].y : sg[k][e].x;
                    rotate_sym(S, Q, A, R);
#pragma unroll
                    for (int e = 0; e < 6; e++) v[k][2 * e + p] = R[e];
                }
                if (DH) {
                    double S[8], R[9];
#pragma unroll
                    for (int e = 0; e < 8; e++) S[e] = p ? sh[k][e].y : sh[k][e].x;
                    rotate_gen(S, Q, A, R);
#pragma unroll
                    for (int e = 0; e < 9; e++) v[k][12 + 2 * e + p] = R[e];
                }
            }
            // formed here, not sunk behind the waits below
#pragma unroll
            for (int e = DG ? 0 : 12; e < (DH ? 2 * kPatchPairs : 12); e++) asm volatile("" : "+v"(v[k][e]));
        }
        wait_for(cleared, kWaves * r);
        wait_for(turns, t);
        const int corner[3] = {ge.x, ge.y, ge.z};
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int slot = (unsigned)corner[k] >> 24;
            const int step = (act >> lane) & 1 ? (ge.w >> (8 * k)) & 0xff : kNoStep;
            const int nsub = (info.z >> (8 * k)) & 0xff;
            in_sub_steps(nsub, step, wave_sync, [&]() __attribute__((always_inline)) {
                // read-modify-write of the slot's words, kRmw reads in flight
#pragma unroll
                for (int e0 = DG ? 0 : 6; e0 < (DH ? kPatchPairs : 6); e0 += kRmw) {
                    double2 u[kRmw];
#pragma unroll
                    for (int e = e0; e < e0 + kRmw && e < (DH ? kPatchPairs : 6); e++) u[e - e0] = acc[e * kPatchVerts + slot];
#pragma unroll
                    for (int e = e0; e < e0 + kRmw && e < (DH ? kPatchPairs : 6); e++)
                        acc[e * kPatchVerts + slot] = make_double2(u[e - e0].x + v[k][2 * e], u[e - e0].y + v[k][2 * e + 1]);
                }
            });
        }
        wave_sync();  // every lane's adds before the turn is given on
        __hip_atomic_store(turns, t + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    while (written < nr) write_row(written++);
}

// BANDED: the distance-banded rule (CQBEM_QUAD_BANDED) is compiled in; without it the tile rule check is not.
template <bool DG, bool DH, bool GAL, bool BANDED>
__global__ void __launch_bounds__(kPatchThreads, 2) k_colloc_gh_patch(Geom g, const double4 *__restrict__ pts, int npts,
                                                                  const Freq *__restrict__ freqs, int l0, Mat m, int row0,
                                                                  const double4 *__restrict__ tpts,
                                                                  const int *__restrict__ patch_chunk,
                                                                  const int4 *__restrict__ chunk_info,
                                                                  const int4 *__restrict__ chunk_faces,
                                                                  const int *__restrict__ patch_verts, cd *__restrict__ UG,
                                                                  cd *__restrict__ UH, long long ld, long long lstride,
                                                                  int nrows, int rpt, int real_hi, Bands bands) {
    __shared__ double2 acc[kPatchPairs * kPatchVerts];      // [word][slot]
    __shared__ double2 frame[kFramePairs * kPatchThreads];
    __shared__ __align__(32) double2 exps[kExpWords];
    auto dest = [=] { return PatchDest{patch_verts, UG, UH, ld, lstride}; };
    const int r0 = blockIdx.z * rpt, nr = min(rpt, nrows - r0);
    auto tile = [&](const auto &f, int l) {
        patch_tile<DG, DH, GAL>(g, pts, npts, BANDED ? bands : Bands{}, f, m, row0, tpts, patch_chunk, chunk_info, chunk_faces, dest,
                                blockIdx.x, l, r0, nr, acc, frame, exps);
    };
    if (real_hi >= 0 && blockIdx.y == 0) tile(point_freq(freqs + l0, real_hi, rp{}), real_hi);
    else if (beyond_table(freqs, l0 + blockIdx.y)) tile(point_freq(freqs, l0 + blockIdx.y, cd{}), blockIdx.y);
    else tile(table_freq(freqs, l0 + blockIdx.y), blockIdx.y);
}

// ------------------------------------------------------------------------
// Several objects' G/H regular-face work in one launch: each piece (an object's row slab) contributes
// npatches x nl x nrows tiles, numbered from its `base`, and each tile runs exactly the computation of
// k_colloc_gh_patch's block for it, so every object's spectra are bit-identical to its own launch.  Two forms:
//   k_scene_gh_tiles: one block per tile; the hardware's workgroup dispatcher hands tiles to CUs in tile order as
//     they free up (pieces are ordered largest first by the host).  Same registers as the single-object kernel
//     plus the piece lookup: 2 waves per SIMD.
//   k_scene_gh_persistent: persistent blocks that take tile numbers from a device counter with one atomic add per tile.
//     The loop-carried state takes it past 256 registers and 80 KB of LDS: one block per CU is resident, of the two per
//     CU that are launched (CQBEM_SCENE_KERNEL=persistent selects it, for comparison).
// ------------------------------------------------------------------------
template <bool DG, bool DH>
__device__ __attribute__((always_inline)) inline void scene_tile(const ScenePiece *__restrict__ pieces, int npieces, unsigned t, double2 *acc, double2 *frame, double2 *exps) {
    int pi = 0;
    while (pi + 1 < npieces && (unsigned)*(const_int *)&pieces[pi + 1].base <= t) ++pi;
    pi = __builtin_amdgcn_readfirstlane(pi);
    ScenePiece P;  // held in scalar registers
    {
        static_assert(sizeof(ScenePiece) % 4 == 0, "copied in words");
        const_int *src = (const_int *)(pieces + pi);
        int w[sizeof(ScenePiece) / 4];
#pragma unroll
        for (unsigned k = 0; k < sizeof(ScenePiece) / 4; k++) w[k] = src[k];
        __builtin_memcpy(&P, w, sizeof(P));
    }
    P.g.V = as_global(P.g.V), P.g.vmap = as_global(P.g.vmap);
    P.bands.sphere = as_global(P.bands.sphere);
    auto dest = [pieces, pi] {
        const ScenePiece *q = pieces + pi;
        asm volatile("" : "+s"(q));
        auto ptr = [](const void *field) { return *(const __attribute__((address_space(4))) unsigned long long *)field; };
        return PatchDest{as_global((const int *)ptr(&q->patch_verts)), as_global((cd *)ptr(&q->UG)), as_global((cd *)ptr(&q->UH)),
                         (long long)ptr(&q->ld), (long long)ptr(&q->lstride)};
    };
    const unsigned local = t - P.base, np = (unsigned)P.npatches, nl = (unsigned)P.slots;
    const unsigned rest = local / np;
    const int pc = __builtin_amdgcn_readfirstlane(local - rest * np), l = __builtin_amdgcn_readfirstlane(rest % nl),
              r0 = __builtin_amdgcn_readfirstlane(rest / nl) * P.rpt;
    auto tile = [&](const auto &f, int lf) {
        patch_tile<DG, DH, false>(P.g, P.pts, P.npts, P.bands, f, P.m, P.row0, nullptr, as_global(P.patch_chunk), P.chunk_info,
                                  as_global(P.chunk_faces), dest, pc, lf, r0, min(P.rpt, P.nrows - r0), acc, frame, exps);
    };
    if (P.real_hi >= 0 && l == 0) tile(point_freq(P.freqs, P.real_hi, rp{}), P.real_hi);
    else if (beyond_table(P.freqs, l)) tile(point_freq(P.freqs, l, cd{}), l);
    else tile(table_freq(P.freqs, l), l);
}

template <bool DG, bool DH>
__global__ void __launch_bounds__(kPatchThreads, 2) k_scene_gh_tiles(const ScenePiece *__restrict__ pieces, int npieces,
                                                                  unsigned t0) {
    __shared__ double2 acc[kPatchPairs * kPatchVerts];
    __shared__ double2 frame[kFramePairs * kPatchThreads];
    __shared__ __align__(32) double2 exps[kExpWords];
    scene_tile<DG, DH>(pieces, npieces, t0 + blockIdx.x, acc, frame, exps);
}

template <bool DG, bool DH>
__global__ void __launch_bounds__(kPatchThreads, 2) k_scene_gh_persistent(const ScenePiece *__restrict__ pieces, int npieces,
                                                                 unsigned ntiles, unsigned *__restrict__ counter) {
    __shared__ double2 acc[kPatchPairs * kPatchVerts];
    __shared__ double2 frame[kFramePairs * kPatchThreads];
    __shared__ __align__(32) double2 exps[kExpWords];
    __shared__ unsigned next_tile;
    for (;;) {
        __syncthreads();  // the previous tile's write-out has read acc; next_tile is free
        if (threadIdx.x == 0) next_tile = atomicAdd(counter, 1u);
        __syncthreads();
        const unsigned t = __builtin_amdgcn_readfirstlane(next_tile);
        if (t >= ntiles) break;  // uniform across the block: every wave leaves
        scene_tile<DG, DH>(pieces, npieces, t, acc, frame, exps);
    }
}

// Zeroes the tile counter of a scene launch (a kernel, not a memset: it is captured in the scene's graph).
__global__ void k_zero_counter(unsigned *counter) {
    if (threadIdx.x == 0) *counter = 0u;
}

// ------------------------------------------------------------------------
// B_trans and B_angular, regular faces.  Grid: (frequency slots, rows), 256 threads: the lanes stride over the faces, then
// the 48 sums are reduced over the lanes and the waves.
//
// Bound by FP64 VALU issue.  A point adds to 12 complex moments of its face
// (h, n.h, h h and two scalars, each times a function of r and s); every factor
// that depends on the frequency alone (1/s^2, s, 1/s) waits until the face's
// or the row's end, and the trace of the h h moment serves as the scalar moment
// of the same function (|h| = 1).  126 instructions per point, 156 beyond the
// reach of the exponentials' table (exp_pair), 203 with the factors applied per point.
// The two real frequencies of an even L share a slot in real arithmetic.
// Icosphere level 4, L = 32: 25.6 ms (31.9 at 156, 33.1 with a slot for each real
// frequency, 43.0 at 203).
// ------------------------------------------------------------------------
constexpr int kBWords = 48;  // B_trans (6 sym complex) + B_angular (18 complex), as doubles

// One lane's sums over its faces: words 2 k, 2 k + 1 of out are entry k, in units of 1/(8 pi s^2).
// GAL: the row is test point tpts[i] (x, y, z, face), whose face's corners are excluded; otherwise vertex i.
// BANDED: each face takes the far rule or the reference rule (a lane then reads its own rule's points; without bands
// they are wave-uniform).
template <bool GAL, bool BANDED, class F>
__device__ __attribute__((always_inline)) inline void b_sums(const Geom &g, const double4 *__restrict__ quad, int npts,
                                                             const F &f, const Mat &m, int i,
                                                             const double4 *__restrict__ tpts,
                                                             const FaceBands &fb, const double2 *exps, double (&out)[kBWords]) {
    typedef typename F::value T;
    double x[3];
    int t[3] = {i, i, i};
    if (GAL) {
        const double4 P = tpts[i];
        x[0] = P.x, x[1] = P.y, x[2] = P.z;
        const int f1 = (int)P.w;
        t[0] = g.F[3 * f1], t[1] = g.F[3 * f1 + 1], t[2] = g.F[3 * f1 + 2];
    } else {
        x[0] = g.V[3 * i], x[1] = g.V[3 * i + 1], x[2] = g.V[3 * i + 2];
    }
    T bt[6], ba[18];  // the row's sums in units of 1/(8 pi s^2)
#pragma unroll
    for (int k = 0; k < 6; k++) bt[k] = T{0, 0};
#pragma unroll
    for (int k = 0; k < 18; k++) ba[k] = T{0, 0};
    for (int fc = threadIdx.x; fc < g.nf; fc += 256) {
        const int c[3] = {g.F[3 * fc], g.F[3 * fc + 1], g.F[3 * fc + 2]};
        if (touches<GAL ? 3 : 1>(g, t, c)) continue;
        // y - x = o + b1 e1 + b2 e2, whose component along the normal is the same at every point
        double o[3], e1[3], e2[3];
        const double n[3] = {g.N[3 * fc], g.N[3 * fc + 1], g.N[3 * fc + 2]};
#pragma unroll
        for (int k = 0; k < 3; k++)
            o[k] = g.V[3 * c[0] + k] - x[k], e1[k] = g.V[3 * c[1] + k] - g.V[3 * c[0] + k], e2[k] = g.V[3 * c[2] + k] - g.V[3 * c[0] + k];
        const double4 *qf = quad;  // the face's rule
        int nq = npts;
        if (BANDED && beyond_sphere(x[0], x[1], x[2], fb.sphere[fc])) qf = fb.far_quad, nq = fb.far_npts;
        T mt[3] = {{0, 0}, {0, 0}, {0, 0}}, m2 = {0, 0}, M[6], S = {0, 0}, S3 = {0, 0};
#pragma unroll
        for (int k = 0; k < 6; k++) M[k] = T{0, 0};
#pragma unroll 1
        for (int q = 0; q < nq; ++q) {
            double b1, b2, w;
            if (BANDED) {
                const double4 Q = qf[q];
                b1 = Q.y, b2 = Q.z, w = Q.w;
            } else {
                const_double *Q = as_const(quad + q);
                b1 = Q[1], b2 = Q[2], w = Q[3];
            }
            double d[3];
#pragma unroll
            for (int k = 0; k < 3; k++) d[k] = fma(b1, e1[k], fma(b2, e2[k], o[k]));
            const double d2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
            const double ir = rsqrt_h3(d2), r = d2 * ir;
            const T z1 = f.sc1 * r, z2 = f.sc2 * r;
            T E1, E2;
            exp_pair(r, z1, z2, f, exps, E1, E2);
            const T s2 = z2 * E2 + E2, dS = (z1 * E1 + E1) - s2;  // s^2 A2, s^2 (A1 - A2)
            const double w2 = (w * ir) * ir, w3 = w2 * ir;
            const double h[3] = {w3 * d[0], w3 * d[1], w3 * d[2]};  // w h / r^2
#pragma unroll
            for (int a = 0; a < 3; a++) {
                fma_cr(mt[a], dS, h[a]);
#pragma unroll
                for (int b = a; b < 3; b++) fma_cr(M[sidx(a, b)], dS, h[a] * d[b]);  // w h h / r
            }
            fma_cr(m2, add_one(s2, -1.0), w3);
            const T v = E2 * m.ic2;
            T u = v;
            fma_cr(u, E1, -m.ic1);
            fma_cr(S, u, w);
            fma_cr(S3, v, w);
        }
        // the face's moments in units of area/s^2; m2 still lacks the normal component of y - x
        const double ar = g.area[fc], rn = o[0] * n[0] + o[1] * n[1] + o[2] * n[2];
        m2 = m2 * (2.0 * rn * ar);
        S = (S * f.s + (M[0] + M[1] + M[2])) * ar, S3 = S3 * f.s * (2.0 * ar);
#pragma unroll
        for (int k = 0; k < 3; k++) mt[k] = mt[k] * ar;
#pragma unroll
        for (int k = 0; k < 6; k++) M[k] = M[k] * ar;
#pragma unroll
        for (int k = 0; k < 3; k++) M[k] += S;  // M_ak + S d_ak: both meet the same normal below
#pragma unroll
        for (int a = 0; a < 3; a++)
#pragma unroll
            for (int b = a; b < 3; b++) {
                T &v = bt[sidx(a, b)];
                fma_cr(v, mt[a], n[b]);
                fma_cr(v, mt[b], n[a]);
                if (a == b) v += m2;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    T &u = ba[sidx(a, b) * 3 + k];
                    fma_cr(u, M[sidx(a, k)], n[b]);
                    fma_cr(u, M[sidx(b, k)], n[a]);
                    if (a == b) fma_cr(u, S3, n[k]);
                }
            }
    }
#pragma unroll
    for (int k = 0; k < 6; k++) out[2 * k] = bt[k].x, out[2 * k + 1] = bt[k].y;
#pragma unroll
    for (int k = 0; k < 18; k++) out[12 + 2 * k] = ba[k].x, out[13 + 2 * k] = ba[k].y;
}

// Sums v over the 64 lanes: lanes 8 j .. 8 j + 7 get the sums of words 6 j .. 6 j + 5 in v[0..5].  Three steps halve the
// words a lane holds (48, 24, 12, 6), the last three add the same 6: 60 exchanges, where 6 steps of 48 words are 288.
__device__ __attribute__((always_inline)) inline void wave_sum48(double (&v)[kBWords], int lane) {
#pragma unroll
    for (int n = 24, o = 32; n >= 6; n /= 2, o /= 2) {
        const bool hi = lane & o;
#pragma unroll
        for (int k = 0; k < n; k++) v[k] = (hi ? v[k + n] : v[k]) + __shfl_xor(hi ? v[k] : v[k + n], o, 64);
    }
#pragma unroll
    for (int o = 4; o > 0; o >>= 1)
#pragma unroll
        for (int k = 0; k < 6; k++) v[k] += __shfl_xor(v[k], o, 64);
}

// GAL: the rows are test points row0 + r, written to rows 3r..3r+2 of an nv3-row buffer; otherwise collocation vertices
// i = row0 + r, written to rows 3i..3i+2.
template <bool GAL, bool BANDED>
__global__ void __launch_bounds__(256, 2) k_colloc_b(Geom g, const double4 *__restrict__ quad, int npts,
                                                   const Freq *__restrict__ freqs, int l0, Mat m, int row0,
                                                   const double4 *__restrict__ tpts, cd *__restrict__ Bt,
                                                   cd *__restrict__ Ba, long long nv3, int real_hi, FaceBands fb) {
    __shared__ double red[4][kBWords];
    __shared__ __align__(32) double2 exps[kExpWords];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = blockIdx.y, slot = blockIdx.x, i = row0 + r;
    const bool real = real_hi >= 0 && slot == 0;
    double v[kBWords];
    auto sums = [&](const auto &f) {
        fill_exp_table(f, exps);
        __syncthreads();
        b_sums<GAL, BANDED>(g, quad, npts, f, m, i, tpts, fb, exps, v);
    };
    if (real) sums(point_freq(freqs + l0, real_hi, rp{}));
    else if (beyond_table(freqs, l0 + slot)) sums(point_freq(freqs, l0 + slot, cd{}));
    else sums(table_freq(freqs, l0 + slot));
    wave_sum48(v, lane);
    if ((lane & 7) == 0) {
#pragma unroll
        for (int k = 0; k < 6; k++) red[wave][6 * (lane >> 3) + k] = v[k];
    }
    __syncthreads();
    if (wave) return;
#pragma unroll
    for (int k = 0; k < 6; k++) {  // the waves' sums, in wave order
        const int w = 6 * (lane >> 3) + k;
        v[k] = (red[0][w] + red[1][w]) + (red[2][w] + red[3][w]);
    }
    const int q = lane & 7;
    if (q > 2) return;
    // one entry per lane; scattered from the packed symmetric form to its full positions
    const int k = 3 * (lane >> 3) + q;
    const double sx = q == 0 ? v[0] : q == 1 ? v[2] : v[4], sy = q == 0 ? v[1] : q == 1 ? v[3] : v[5];
    cd e0, e1{0, 0};  // the entry at frequency slot, or the two real entries at frequencies 0 and real_hi
    if (real) {
        const PointFreq<rp> f = point_freq(freqs + l0, real_hi, rp{});
        e0 = cd{sx * f.is2.x * kInv8Pi, 0.0}, e1 = cd{sy * f.is2.y * kInv8Pi, 0.0};
    } else {
        e0 = cd{sx, sy} * point_freq(freqs, l0 + slot, cd{}).is2 * kInv8Pi;
    }
    const int io = GAL ? r : i, words = k < 6 ? 3 : 9;
    const int ab = k < 6 ? k : (k - 6) / 3, c = k < 6 ? 0 : (k - 6) % 3;
    cd *o = (k < 6 ? Bt : Ba) + (long long)(3 * io) * words;
    for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++)
            if (sidx(a, b) == ab) {
                cd *p = o + a * words + (k < 6 ? b : 3 * b + c);
                p[slot * nv3 * words] = e0;
                if (real) p[real_hi * nv3 * words] = e1;
            }
}

// ------------------------------------------------------------------------
// Singular faces (faces touching the collocation vertex).  One lane per
// (row vertex, frequency); the lane owns those rows and adds into them.
//   KIND 0: G, weakly singular polar rule (integrator_collocation.hpp:19-63)
//   KIND 1: B_trans + B_angular, same polar rule
//   KIND 2: H, Guiggiani finite-part rule (integrator_collocation.hpp:65-124)
// ------------------------------------------------------------------------
constexpr int kSingMaxFaces = 16;  // singular faces per batch of one (row, frequency) wavefront

// Sums v over the groups of gs lanes, in lane order: sum[group][k] for the first ngroups groups.  Through LDS, 9 words of
// every lane at a time, each sum taken by one lane; a single wave per block.  (By shuffles, each lane read its gs - 1
// successors' words: 36 cross-lane moves per entry at gs = 10.)
template <int N, int NE>
__device__ __attribute__((always_inline)) inline void group_sums(const cd (&v)[N], cd (*sum)[NE], cd (*part)[64], int lane, int gs, int ngroups) {
#pragma unroll
    for (int k0 = 0; k0 < N; k0 += 9) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 9; k++)
            if (k0 + k < N) part[k][lane] = v[k0 + k];
        __syncthreads();
        const int n = N - k0 < 9 ? N - k0 : 9;
        for (int o = lane; o < n * ngroups; o += 64) {
            const int grp = o / n, k = o - grp * n;
            cd t = part[k][grp * gs];
            for (int q = 1; q < gs; q++) t += part[k][grp * gs + q];
            sum[grp][k0 + k] = t;
        }
    }
    __syncthreads();
}

__device__ inline void unit3(double v[3]) {
    const double n = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
    if (n > 0) v[0] /= n, v[1] /= n, v[2] /= n;
}

template <int KIND>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) k_colloc_singular(Geom g, const double2 *__restrict__ line, int nline,
                                                         const Freq *__restrict__ freqs, int l0, int nl, Mat m, int row0,
                                                         int nrows, cd *__restrict__ U, long long ld, long long lstride,
                                                         cd *__restrict__ Bt, cd *__restrict__ Ba, long long nv3) {
    constexpr int NE = KIND == 1 ? 36 : 27;  // per face: B 9 + 27 entries; G/H 3 corners x 3 x 3
    __shared__ cd fsum[kSingMaxFaces][NE], part[9][64];
    __shared__ int fj[kSingMaxFaces][3], umap[kSingMaxFaces][3], ucol[3 * kSingMaxFaces + 1];
    const int il = blockIdx.x / nl, l = blockIdx.x % nl;
    const int i = row0 + il;
    const Freq f = freqs[l0 + l];
    // GS lanes per singular face, lane t of a group takes the angular points t, t + GS, ...
    const int GS = nline < 64 / kSingMaxFaces ? 64 / kSingMaxFaces : (nline > 64 ? 64 : nline);
    const int FB = 64 / GS;  // faces per batch
    const int lane = threadIdx.x, slot = lane / GS, t = lane % GS;
    const int fbeg = g.sg_ptr[i], fend = g.sg_ptr[i + 1];
    for (int fb = fbeg; fb < fend; fb += FB) {
        const int nb = min(FB, fend - fb);
        const bool active = slot < nb;
        const int pk = g.sg_face[active ? fb + slot : fbeg];
        const int fc = pk >> 2, c = pk & 3;
        const int j[3] = {g.F[3 * fc + c], g.F[3 * fc + (c + 1) % 3], g.F[3 * fc + (c + 2) % 3]};
        double y1[3], y2[3], y3[3], n[3];
        for (int k = 0; k < 3; k++)
            y1[k] = g.V[3 * j[0] + k], y2[k] = g.V[3 * j[1] + k], y3[k] = g.V[3 * j[2] + k], n[k] = g.N[3 * fc + k];
        double v1[3], v2[3];
        for (int k = 0; k < 3; k++) v1[k] = y2[k] - y1[k], v2[k] = y3[k] - y1[k];
        const bool leader = active && t == 0;  // turns the face's sums (group_sums) into its entries
        if (KIND == 0 || KIND == 1) {
            // polar frame around y1
            double u1[3] = {v1[0], v1[1], v1[2]}, u2[3] = {v2[0], v2[1], v2[2]};
            unit3(u1), unit3(u2);
            const double xh[3] = {u1[0], u1[1], u1[2]};
            double cxu[3] = {xh[1] * u2[2] - xh[2] * u2[1], xh[2] * u2[0] - xh[0] * u2[2], xh[0] * u2[1] - xh[1] * u2[0]};
            double yh[3] = {cxu[1] * xh[2] - cxu[2] * xh[1], cxu[2] * xh[0] - cxu[0] * xh[2], cxu[0] * xh[1] - cxu[1] * xh[0]};
            unit3(yh);
            double e[3] = {v1[0] - v2[0], v1[1] - v2[1], v1[2] - v2[2]};
            unit3(e);
            const double d = v1[0] * e[0] + v1[1] * e[1] + v1[2] * e[2];
            double v12[3] = {v1[0] - d * e[0], v1[1] - d * e[1], v1[2] - d * e[2]};
            const double a = sqrt(v12[0] * v12[0] + v12[1] * v12[1] + v12[2] * v12[2]);
            unit3(v12);
            const double alpha = acos(u1[0] * u2[0] + u1[1] * u2[1] + u1[2] * u2[2]);
            // beta = angle(v12, u1), which the reference takes as acos of the clamped dot product
            // (integrator_collocation.hpp:36); atan2(|v12 x u1|, v12 . u1) is the same angle without acos's
            // loss of half the digits near 0 (a right angle at y2, common on cube meshes)
            const double bx = v12[1] * u1[2] - v12[2] * u1[1], by = v12[2] * u1[0] - v12[0] * u1[2],
                         bz = v12[0] * u1[1] - v12[1] * u1[0];
            const double beta = atan2(sqrt(bx * bx + by * by + bz * bz), v12[0] * u1[0] + v12[1] * u1[1] + v12[2] * u1[2]);
            // barycentric projection setup (barycentric_coordinates.cuh:15-38)
            const double d00 = v1[0] * v1[0] + v1[1] * v1[1] + v1[2] * v1[2];
            const double d01 = v1[0] * v2[0] + v1[1] * v2[1] + v1[2] * v2[2];
            const double d11 = v2[0] * v2[0] + v2[1] * v2[1] + v2[2] * v2[2];
            const double iden = 1.0 / (d00 * d11 - d01 * d01);
            cd ga[3][6], gb[3];
            cd mt[3], m2, M[6], S, S3;
            if (KIND == 0) {
                for (int k = 0; k < 3; k++) {
                    gb[k] = cd{0, 0};
                    for (int e2 = 0; e2 < 6; e2++) ga[k][e2] = cd{0, 0};
                }
            } else {
                for (int k = 0; k < 3; k++) mt[k] = cd{0, 0};
                for (int k = 0; k < 6; k++) M[k] = cd{0, 0};
                m2 = S = S3 = cd{0, 0};
            }
            for (int it = active ? t : nline; it < nline; it += GS) {
                const double th = alpha * line[it].x, wth = alpha * line[it].y;
                double sth, cth;
                sincos(th, &sth, &cth);
                const double h[3] = {xh[0] * cth + yh[0] * sth, xh[1] * cth + yh[1] * sth, xh[2] * cth + yh[2] * sth};
                const double rmax = a / cos(th - beta);
                const double rn = h[0] * n[0] + h[1] * n[1] + h[2] * n[2];
                for (int ir_ = 0; ir_ < nline; ++ir_) {
                    const double r = rmax * line[ir_].x, w = wth * rmax * line[ir_].y;
                    const double ir = 1.0 / r, ir2 = ir * ir;
                    const Expo E = expo(r, f);
                    if (KIND == 0) {
                        // clamped projection barycentrics of y = y1 + r h
                        const double c0 = r * h[0], c1 = r * h[1], c2 = r * h[2];
                        const double d20 = c0 * v1[0] + c1 * v1[1] + c2 * v1[2];
                        const double d21 = c0 * v2[0] + c1 * v2[1] + c2 * v2[2];
                        double L1 = (d11 * d20 - d01 * d21) * iden, L2 = (d00 * d21 - d01 * d20) * iden;
                        double L0 = 1.0 - (L1 + L2);
                        L0 = fmin(1.0, fmax(0.0, L0)), L1 = fmin(1.0, fmax(0.0, L1)), L2 = fmin(1.0, fmax(0.0, L2));
                        const double Lb[3] = {L0, L1, L2};
                        cd al, be;
                        g_coef(E, ir, ir2, m, al, be);  // r * u_hat coefficients
                        for (int k = 0; k < 3; k++) {
                            const double wk = w * Lb[k];
                            const cd ak = al * wk;
                            fma_cr(gb[k], be, wk);
                            fma_cr(ga[k][0], ak, h[0] * h[0]);
                            fma_cr(ga[k][1], ak, h[1] * h[1]);
                            fma_cr(ga[k][2], ak, h[2] * h[2]);
                            fma_cr(ga[k][3], ak, h[0] * h[1]);
                            fma_cr(ga[k][4], ak, h[0] * h[2]);
                            fma_cr(ga[k][5], ak, h[1] * h[2]);
                        }
                    } else {
                        cd t1, t2, u1c, u12, u3;
                        b_coef(E, ir, ir2, f, m, t1, t2, u1c, u12, u3);
                        const double wr = w * r;  // polar rules integrate r * kernel
                        t1 = t1 * wr;
                        u1c = u1c * wr;
                        for (int a2 = 0; a2 < 3; a2++) fma_cr(mt[a2], t1, h[a2]);
                        fma_cr(m2, t2, wr * rn);
                        for (int a2 = 0; a2 < 3; a2++)
                            for (int b = a2; b < 3; b++) fma_cr(M[sidx(a2, b)], u1c, h[a2] * h[b]);
                        fma_cr(S, u12, wr);
                        fma_cr(S3, u3, wr);
                    }
                }
            }
            if (KIND == 0) {
                cd v[21];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    v[7 * k + 6] = gb[k];
#pragma unroll
                    for (int e2 = 0; e2 < 6; e2++) v[7 * k + e2] = ga[k][e2];
                }
                group_sums(v, fsum, part, lane, GS, nb);
                if (leader) {
#pragma unroll
                    for (int k = 0; k < 21; k++) v[k] = fsum[slot][k];
#pragma unroll
                    for (int k = 0; k < 3; k++)
#pragma unroll
                        for (int a2 = 0; a2 < 3; a2++)
#pragma unroll
                            for (int b = 0; b < 3; b++) {
                                cd u = v[7 * k + sidx(a2, b)];
                                if (a2 == b) u += v[7 * k + 6];
                                fsum[slot][k * 9 + a2 * 3 + b] = u;
                            }
                }
            } else {
                cd v12s[12] = {mt[0], mt[1], mt[2], M[0], M[1], M[2], M[3], M[4], M[5], m2, S, S3};
                group_sums(v12s, fsum, part, lane, GS, nb);
                if (leader) {
                    for (int k = 0; k < 3; k++) mt[k] = fsum[slot][k];
                    for (int k = 0; k < 6; k++) M[k] = fsum[slot][3 + k];
                    m2 = fsum[slot][9], S = fsum[slot][10], S3 = fsum[slot][11];
                }
                if (leader)
                for (int a2 = 0; a2 < 3; a2++)
                    for (int b = 0; b < 3; b++) {
                        cd v = {0, 0};
                        fma_cr(v, mt[a2], n[b]);
                        fma_cr(v, mt[b], n[a2]);
                        if (a2 == b) v += m2;
                        fsum[slot][a2 * 3 + b] = v;
                        for (int k = 0; k < 3; k++) {
                            cd u = {0, 0};
                            fma_cr(u, M[sidx(a2, k)], n[b]);
                            fma_cr(u, M[sidx(b, k)], n[a2]);
                            fma_cr(u, S, (b == k ? n[a2] : 0.0) + (a2 == k ? n[b] : 0.0));
                            if (a2 == b) fma_cr(u, S3, n[k]);
                            fsum[slot][9 + a2 * 9 + b * 3 + k] = u;
                        }
                    }
            }
        } else {
            // Guiggiani: rho-theta on the unit right triangle around y1
            double cr[3] = {v1[1] * v2[2] - v1[2] * v2[1], v1[2] * v2[0] - v1[0] * v2[2], v1[0] * v2[1] - v1[1] * v2[0]};
            const double J = sqrt(cr[0] * cr[0] + cr[1] * cr[1] + cr[2] * cr[2]);
            cd out[27];
            for (int k = 0; k < 27; k++) out[k] = cd{0, 0};
            const double half_pi = 1.5707963267948966192;
            for (int it = active ? t : nline; it < nline; it += GS) {
                const double th = half_pi * line[it].x, wth = half_pi * line[it].y;
                double st, ct;
                sincos(th, &st, &ct);
                double Av[3] = {ct * v1[0] + st * v2[0], ct * v1[1] + st * v2[1], ct * v1[2] + st * v2[2]};
                const double A = sqrt(Av[0] * Av[0] + Av[1] * Av[1] + Av[2] * Av[2]);
                const double Ah[3] = {Av[0] / A, Av[1] / A, Av[2] / A};
                const double rho_bar = 1.0 / (cos(th - 0.78539816339744830962) * 1.4142135623730950488);
                const double rn = Ah[0] * n[0] + Ah[1] * n[1] + Ah[2] * n[2];
                // cancelling term f_pq = (1/4pi) kap (Ah_p n_q - Ah_q n_p) / A^2 * J, basis (1,0,0)
                const double fs = kInv4Pi * m.kap * J / (A * A);
                cd S1[3], S2[3], S4[3];
                for (int k = 0; k < 3; k++) S1[k] = S2[k] = S4[k] = cd{0, 0};
                double sinv = 0.0;
                for (int ir_ = 0; ir_ < nline; ++ir_) {
                    const double rho = rho_bar * line[ir_].x, w = rho_bar * line[ir_].y;
                    const double r = rho * A;
                    const double ir = 1.0 / r, ir2 = ir * ir;
                    const Expo E = expo(r, f);
                    cd c1, c2, c4;
                    h_coef(E, ir, ir2, f, m, c1, c2, c4);
                    const double Lb[3] = {1.0 - rho * (ct + st), rho * ct, rho * st};
                    for (int k = 0; k < 3; k++) {
                        const double wk = w * Lb[k] * J * rho;
                        fma_cr(S1[k], c1, wk);
                        fma_cr(S2[k], c2, wk);
                        fma_cr(S4[k], c4, wk);
                    }
                    sinv += w / rho;
                }
                const double lg = log(rho_bar * A);
                for (int p = 0; p < 3; p++)
                    for (int qq = 0; qq < 3; qq++) {
                        const double fpq = fs * (Ah[p] * n[qq] - Ah[qq] * n[p]);
                        for (int k = 0; k < 3; k++) {
                            cd v = {0, 0};
                            fma_cr(v, S1[k], Ah[p] * n[qq]);
                            fma_cr(v, S2[k], n[p] * Ah[qq] + (p == qq ? rn : 0.0));
                            fma_cr(v, S4[k], rn * Ah[p] * Ah[qq]);
                            v = v * kInv4Pi;
                            if (k == 0) v.x += fpq * (lg - sinv);
                            fma_cr(out[(p * 3 + qq) * 3 + k], v, wth);
                        }
                    }
            }
            cd v[27];  // in fsum's order
#pragma unroll
            for (int e = 0; e < 9; e++)
#pragma unroll
                for (int k = 0; k < 3; k++) v[k * 9 + e] = out[e * 3 + k];
            group_sums(v, fsum, part, lane, GS, nb);
        }
        if (leader)
            for (int k = 0; k < 3; k++) fj[slot][k] = j[k];
        __syncthreads();
        // add the batch's faces into the row: each output entry sums its faces in face order, then one
        // read-modify-write per entry (no dependent chains through memory)
        if (KIND == 1) {
            if (lane < 36) {
                cd sum = fsum[0][lane];
                for (int s2 = 1; s2 < nb; s2++) sum += fsum[s2][lane];
                cd *o = lane < 9 ? Bt + (long long)l * nv3 * 3 + (long long)(3 * i) * 3 + lane
                                 : Ba + (long long)l * nv3 * 9 + (long long)(3 * i) * 9 + (lane - 9);
                *o += sum;
            }
        } else {
            // distinct columns of the batch in order of first appearance
            if (lane == 0) {
                int nu = 0;
                for (int s2 = 0; s2 < nb; s2++)
                    for (int k = 0; k < 3; k++) {
                        int u = 0;
                        while (u < nu && ucol[u] != fj[s2][k]) u++;
                        if (u == nu) ucol[nu++] = fj[s2][k];
                        umap[s2][k] = u;
                    }
                ucol[3 * kSingMaxFaces] = nu;
            }
            __syncthreads();
            const int nu = ucol[3 * kSingMaxFaces];
            for (int item = lane; item < 9 * nu; item += 64) {
                const int u = item / 9, e = item % 9, a2 = e / 3, b = e % 3;
                cd sum = {0, 0};
                for (int s2 = 0; s2 < nb; s2++)
                    for (int k = 0; k < 3; k++)
                        if (umap[s2][k] == u) sum += fsum[s2][k * 9 + e];
                U[(long long)l * lstride + (long long)(3 * il + a2) * ld + 3 * (long long)ucol[u] + b] += sum;
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------
// Inverse CQ transform: W_n[e] = sum_l Re(X_l[e] * T[n][l]), with the table
// T[n][l] = R^-n / L * mult_l * zeta^(-n l) (G.cu:166-179).  One lane per
// entry, NC weights per pass; the table index is uniform (scalar loads).
// ------------------------------------------------------------------------
// Inverse CQ transform of one chunk of NC weights n0 .. n0+NC-1: out[n][e] = sum_l Re(X_l(e) T(n, l)), with
// T(n, l) = (2 or 1) R^-n / L exp(-2 pi i n l / L) (the half-spectrum table).  The chunk's table lives in LDS (read as
// broadcasts) and the spectrum is read LC frequencies at a time so that their loads are in flight together.
constexpr int kTransformNC = 32, kTransformMaxLf = 64;

// OutT: double, or float for resident weights stored in single precision (the sum is formed in double and rounded once).
// Two adjacent entries per lane (ALIGNED: E and out_nstride even, out aligned to a pair; otherwise the stores are
// declared unaligned and an odd E's last entry is alone): each
// frequency's two complex values in one 32-byte read, each weight's two values in one 16-byte store (the store
// width HBM writes best), and a grid that covers every pair at once.  Each weight is the same sum, term for
// term.  LC = 2 frequencies per batch of loads keeps the kernel within 168 VGPRs: 3 waves per SIMD (with 4 it takes
// 181 VGPRs and 2 waves, 2.6% slower).
typedef double d2v __attribute__((ext_vector_type(2)));
typedef float f2v __attribute__((ext_vector_type(2)));
template <class OutT> struct Pair2;
template <> struct Pair2<double> {
    typedef d2v type;
};
template <> struct Pair2<float> {
    typedef f2v type;
};
template <int LC, bool ALIGNED, class OutT>
__global__ void __launch_bounds__(256, 3) k_transform_pair(const cd *__restrict__ spec, long long E, long long spec_ls, int Lf,
                                                        const double2 *__restrict__ tab, int L, int n0,
                                                        OutT *__restrict__ out, long long out_nstride) {
    constexpr int NC = kTransformNC;
    __shared__ double2 T[NC * kTransformMaxLf];  // [l][k]
    for (int t = threadIdx.x; t < NC * Lf; t += 256) {
        const int l = t / NC, k = t % NC;
        T[t] = n0 + k < L ? tab[(long long)(n0 + k) * Lf + l] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * 2;
    if (e >= E) return;
    double a0[NC], a1[NC];
#pragma unroll
    for (int k = 0; k < NC; k++) a0[k] = a1[k] = 0.0;
    for (int l0 = 0; l0 < Lf; l0 += LC) {
        d2v X0[LC], X1[LC];
#pragma unroll
        for (int c = 0; c < LC; c++) {
            // each spectrum value is read once: streaming (non-temporal) loads
            const d2v *src = reinterpret_cast<const d2v *>(spec + (long long)(l0 + c) * spec_ls + e);
            if (l0 + c < Lf) {
                X0[c] = __builtin_nontemporal_load(src);
                X1[c] = ALIGNED || e + 1 < E ? __builtin_nontemporal_load(src + 1) : d2v{0.0, 0.0};
            } else {
                X0[c] = d2v{0.0, 0.0}, X1[c] = d2v{0.0, 0.0};
            }
        }
#pragma unroll
        for (int c = 0; c < LC; c++) {
            if (l0 + c >= Lf) break;
            const double2 *Tl = T + (l0 + c) * NC;
#pragma unroll
            for (int k = 0; k < NC; k++) {
                a0[k] = fma(X0[c].x, Tl[k].x, fma(-X0[c].y, Tl[k].y, a0[k]));
                a1[k] = fma(X1[c].x, Tl[k].x, fma(-X1[c].y, Tl[k].y, a1[k]));
            }
        }
    }
    typedef typename Pair2<OutT>::type V2;
#pragma unroll
    for (int k = 0; k < NC; k++) {
        const int n = n0 + k;
        if (n < L) {
            typedef V2 V2u __attribute__((aligned(sizeof(OutT))));
            const V2 w = {(OutT)a0[k], (OutT)a1[k]};
            OutT *o = out + (long long)n * out_nstride + e;  // written once
            if (ALIGNED) __builtin_nontemporal_store(w, reinterpret_cast<V2 *>(o));
            else if (e + 1 < E) __builtin_nontemporal_store(w, reinterpret_cast<V2u *>(o));
            else __builtin_nontemporal_store(w.x, o);
        }
    }
}

// Same for Lf > kTransformMaxLf, with the table read from global memory.
template <int NC, class OutT>
__global__ void __launch_bounds__(256) k_transform_wide(const cd *__restrict__ spec, long long E, long long spec_ls, int Lf,
                                                         const double2 *__restrict__ tab, int L, int n0,
                                                         OutT *__restrict__ out, long long out_nstride) {
    const long long stride = (long long)gridDim.x * 256;
    for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < E; e += stride) {
        double acc[NC];
#pragma unroll
        for (int k = 0; k < NC; k++) acc[k] = 0.0;
        for (int l = 0; l < Lf; l++) {
            const cd X = spec[(long long)l * spec_ls + e];
#pragma unroll
            for (int k = 0; k < NC; k++) {
                const int n = n0 + k;
                if (n < L) {
                    const double2 Tv = tab[(long long)n * Lf + l];
                    acc[k] = fma(X.x, Tv.x, fma(-X.y, Tv.y, acc[k]));
                }
            }
        }
#pragma unroll
        for (int k = 0; k < NC; k++) {
            const int n = n0 + k;
            if (n < L) out[(long long)n * out_nstride + e] = (OutT)acc[k];
        }
    }
}

// ------------------------------------------------------------------------
// History term of one CQ time step on the resident matrices:
//   b = sum_{i=1..m} (G_i p[nh-i] - H_i u[nh-i] + B_i acc[nh-i]).
// One wavefront per row; lanes stride the columns with kHistUnroll independent loads per matrix in
// flight (the 2 (L-1) row streams are read once, HBM-bound); fixed-order wave reduction.
// ------------------------------------------------------------------------
constexpr int kHistUnroll = 4;

template <bool HG, bool HH>
__device__ inline double history_row(const double *__restrict__ gr, const double *__restrict__ hr, const double *__restrict__ pv,
                                     const double *__restrict__ uv, long long n3, int lane, double s) {
    long long c = lane;
    for (; c + 64 * (kHistUnroll - 1) < n3; c += 64 * kHistUnroll) {
        double g[kHistUnroll], h[kHistUnroll], x[kHistUnroll], y[kHistUnroll];
#pragma unroll
        for (int k = 0; k < kHistUnroll; k++) {
            if (HG) g[k] = gr[c + 64 * k], x[k] = pv[c + 64 * k];
            if (HH) h[k] = hr[c + 64 * k], y[k] = uv[c + 64 * k];
        }
#pragma unroll
        for (int k = 0; k < kHistUnroll; k++) {
            if (HG) s = fma(g[k], x[k], s);
            if (HH) s = fma(-h[k], y[k], s);
        }
    }
    for (; c < n3; c += 64) {
        if (HG) s = fma(gr[c], pv[c], s);
        if (HH) s = fma(-hr[c], uv[c], s);
    }
    return s;
}

template <bool HG, bool HH>
__global__ void __launch_bounds__(256) k_history(const double *__restrict__ G, const double *__restrict__ H,
                                                  const double *__restrict__ B, const double *__restrict__ p,
                                                  const double *__restrict__ u, const double *__restrict__ acc,
                                                  long long n3, int m, int nh, double *__restrict__ b) {
    const long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= n3) return;
    double s = 0.0;
    for (int i = 1; i <= m; i++) {
        const long long ro = (long long)i * n3 * n3 + r * n3;
        s = history_row<HG, HH>(HG ? G + ro : nullptr, HH ? H + ro : nullptr, HG ? p + (long long)(nh - i) * n3 : nullptr,
                                HH ? u + (long long)(nh - i) * n3 : nullptr, n3, lane, s);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) {
        if (B)
            for (int i = 1; i <= m; i++) {
                const double *br = B + ((long long)i * n3 + r) * 6, *av = acc + (long long)(nh - i) * 6;
#pragma unroll
                for (int k = 0; k < 6; k++) s = fma(br[k], av[k], s);
            }
        b[r] = s;
    }
}

// The same history sum in 16-byte loads.  A16: n3 is even and the matrices and vectors are 16-byte aligned (every row then
// starts on a 16-byte boundary); otherwise the loads are declared 8-byte aligned, which the hardware takes at the price
// of one more cache line per 1 KB, and an odd n3's last column is added on its own: n3 = 3489, 16 steps (3.1 GB) 530 us
// (5.9 TB/s; 709 us in 8-byte loads, one row per wavefront).  SPLIT: history_split.  Each wavefront takes R consecutive rows, so a chunk of p and u loaded once serves R matrix rows
// (the vectors are re-read from L2 by every wavefront: with one row per wavefront that traffic equals the matrix
// stream).  The matrix rows are streamed with 16-byte non-temporal loads: each weight is read once per step.  The
// B terms are spread over the lanes before the wave reduction.  Matrix i starts at G + i * mat_stride (n3^2 for the
// history; 0 with m = nh = 1 makes it y = A x).
typedef double hist_d2 __attribute__((ext_vector_type(2)));
typedef hist_d2 hist_d2u __attribute__((aligned(8)));
typedef float hist_f2 __attribute__((ext_vector_type(2)));
template <class S, bool A16> struct HistPair;
template <> struct HistPair<double, true> { typedef hist_d2 type, vec; };
template <> struct HistPair<double, false> { typedef hist_d2u type, vec; };
template <> struct HistPair<float, true> { typedef hist_f2 type; typedef hist_d2 vec; };

// S: the matrices' element type (double, or float for weights stored in single precision; the products and
// sums are formed in double either way).
template <class S, bool A16, bool SPLIT, bool HG, bool HH, int R>
__global__ void __launch_bounds__(256) k_history_v2(const S *__restrict__ G, const S *__restrict__ H,
                                                     const double *__restrict__ B, const double *__restrict__ p,
                                                     const double *__restrict__ u, const double *__restrict__ acc,
                                                     long long n3, long long mat_stride, int m, int nh,
                                                     double *__restrict__ b) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long r0 = (SPLIT ? (long long)blockIdx.x : (long long)blockIdx.x * 4 + wave) * R;
    if (r0 >= n3) return;  // SPLIT: of the whole block
    const long long nc = n3 >> 1;  // 16-byte columns
    long long rr[R];
#pragma unroll
    for (int k = 0; k < R; k++) rr[k] = r0 + k < n3 ? r0 + k : n3 - 1;  // rows past the end repeat the last (unused)
    double s[R];
#pragma unroll
    for (int k = 0; k < R; k++) s[k] = 0.0;
    for (int i = SPLIT ? 1 + wave : 1; i <= m; i += SPLIT ? 4 : 1) {
        const long long mo = (long long)i * mat_stride;
        typedef typename HistPair<S, A16>::type s2;
        typedef typename HistPair<S, A16>::vec x2;
        const x2 *xp = HG ? reinterpret_cast<const x2 *>(p + (long long)(nh - i) * n3) : nullptr;
        const x2 *xu = HH ? reinterpret_cast<const x2 *>(u + (long long)(nh - i) * n3) : nullptr;
        const s2 *gr[R], *hr[R];
#pragma unroll
        for (int k = 0; k < R; k++) {
            gr[k] = HG ? reinterpret_cast<const s2 *>(G + mo + rr[k] * n3) : nullptr;
            hr[k] = HH ? reinterpret_cast<const s2 *>(H + mo + rr[k] * n3) : nullptr;
        }
        long long c = lane;
        for (; c + 64 * (kHistUnroll - 1) < nc; c += 64 * kHistUnroll) {
            hist_d2 x[kHistUnroll], y[kHistUnroll];
            s2 g[R][kHistUnroll], h[R][kHistUnroll];
#pragma unroll
            for (int j = 0; j < kHistUnroll; j++) {
                if (HG) x[j] = xp[c + 64 * j];
                if (HH) y[j] = xu[c + 64 * j];
#pragma unroll
                for (int k = 0; k < R; k++) {
                    if (HG) g[k][j] = __builtin_nontemporal_load(gr[k] + c + 64 * j);
                    if (HH) h[k][j] = __builtin_nontemporal_load(hr[k] + c + 64 * j);
                }
            }
#pragma unroll
            for (int j = 0; j < kHistUnroll; j++)
#pragma unroll
                for (int k = 0; k < R; k++) {
                    if (HG) s[k] = fma((double)g[k][j].y, x[j].y, fma((double)g[k][j].x, x[j].x, s[k]));
                    if (HH) s[k] = fma(-(double)h[k][j].y, y[j].y, fma(-(double)h[k][j].x, y[j].x, s[k]));
                }
        }
        // the last, partial step: all its loads before the first product
        {
            x2 x[kHistUnroll], y[kHistUnroll];
            s2 g[R][kHistUnroll], h[R][kHistUnroll];
#pragma unroll
            for (int j = 0; j < kHistUnroll; j++)
                if (c + 64 * j < nc) {
                    if (HG) x[j] = xp[c + 64 * j];
                    if (HH) y[j] = xu[c + 64 * j];
#pragma unroll
                    for (int k = 0; k < R; k++) {
                        if (HG) g[k][j] = __builtin_nontemporal_load(gr[k] + c + 64 * j);
                        if (HH) h[k][j] = __builtin_nontemporal_load(hr[k] + c + 64 * j);
                    }
                }
#pragma unroll
            for (int j = 0; j < kHistUnroll; j++)
                if (c + 64 * j < nc) {
#pragma unroll
                    for (int k = 0; k < R; k++) {
                        if (HG) s[k] = fma((double)g[k][j].y, x[j].y, fma((double)g[k][j].x, x[j].x, s[k]));
                        if (HH) s[k] = fma(-(double)h[k][j].y, y[j].y, fma(-(double)h[k][j].x, y[j].x, s[k]));
                    }
                }
        }
        if (!A16 && (n3 & 1) && lane == 0) {  // the last column
            const double x = HG ? p[(long long)(nh - i) * n3 + n3 - 1] : 0.0, y = HH ? u[(long long)(nh - i) * n3 + n3 - 1] : 0.0;
#pragma unroll
            for (int k = 0; k < R; k++) {
                if (HG) s[k] = fma((double)G[mo + rr[k] * n3 + n3 - 1], x, s[k]);
                if (HH) s[k] = fma(-(double)H[mo + rr[k] * n3 + n3 - 1], y, s[k]);
            }
        }
    }
    if (B)
        for (int j = SPLIT ? (int)threadIdx.x : lane; j < 6 * m; j += SPLIT ? 256 : 64) {
            const int i = j / 6 + 1, q = j - 6 * (i - 1);
            const double a = acc[(long long)(nh - i) * 6 + q];
#pragma unroll
            for (int k = 0; k < R; k++) s[k] = fma(B[((long long)i * n3 + rr[k]) * 6 + q], a, s[k]);
        }
#pragma unroll
    for (int k = 0; k < R; k++)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s[k] += __shfl_xor(s[k], o, 64);
    if (SPLIT) {  // the waves' sums, in wave order
        __shared__ double part[4][R];
        if (lane == 0)
#pragma unroll
            for (int k = 0; k < R; k++) part[wave][k] = s[k];
        __syncthreads();
        const int k = threadIdx.x;
        if (k < R && r0 + k < n3) b[r0 + k] = (part[0][k] + part[1][k]) + (part[2][k] + part[3][k]);
        return;
    }
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < R; k++)
            if (r0 + k < n3) b[r0 + k] = s[k];
}

// y = A x for a row-major n x n matrix (u_p p of a constrained time step); one wavefront per row, as k_history.
__global__ void __launch_bounds__(256) k_matvec(const double *__restrict__ A, const double *__restrict__ x, long long n,
                                                double *__restrict__ y) {
    const long long r = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= n) return;
    double s = history_row<true, false>(A + r * n, nullptr, x, nullptr, n, lane, 0.0);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) y[r] = s;
}

// H_0 += C on the 3x3 diagonal blocks (collocation, H.cu:186-191).
template <class T>
__global__ void k_add_c_colloc(T *H0, const double *C, int nv) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= 9 * nv) return;
    const int v = t / 9, a = (t % 9) / 3, b = t % 3;
    const long long n3 = 3LL * nv;
    T &h = H0[(3LL * v + a) * n3 + 3 * v + b];
    h = (T)((double)h + C[t]);
}

// H_0 += C for Galerkin: sparse (row, col, value) triplets, one lane each, rows unique per launch.
template <class T>
__global__ void k_add_triplets(T *H0, const long long *idx, const double *val, long long n) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    H0[idx[t]] = (T)((double)H0[idx[t]] + val[t]);
}

// B_angular += B_trans (x) x_v and B = [B_trans | B_euler] (B_angular.cu:167-175, matrix_collection.cpp:280-305).
__global__ void k_b_post(double *Bt, double *Ba, double *B6, const double *V, int nv, int L) {
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long nr = 3LL * nv;
    if (t >= nr * L) return;
    const long long n = t / nr, r = t % nr;
    const double *bt = Bt + (n * nr + r) * 3;
    double *ba = Ba + (n * nr + r) * 9;
    const double *x = V + 3 * (r / 3);
    for (int j = 0; j < 3; j++)
        for (int k = 0; k < 3; k++) ba[j * 3 + k] += bt[j] * x[k];
    if (B6) {
        double *b6 = B6 + (n * nr + r) * 6;
        for (int j = 0; j < 3; j++) b6[j] = bt[j];
        for (int j = 0; j < 3; j++) b6[3 + j] = ba[((j + 2) % 3) * 3 + (j + 1) % 3] - ba[((j + 1) % 3) * 3 + (j + 2) % 3];
    }
}

// ------------------------------------------------------------- launchers --
hipError_t launch_colloc_gh(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, const Mat &m,
                            int row0, int nrows, cd *UG, cd *UH, long long ld, long long lstride, hipStream_t st) {
    dim3 grid((g.nv + 63) / 64, nl, nrows);
    if (UG && UH)
        hipLaunchKernelGGL((k_colloc_gh<true, true>), grid, dim3(64), 0, st, g, quad, npts, freqs, l0, m, row0, UG, UH, ld,
                           lstride);
    else if (UG)
        hipLaunchKernelGGL((k_colloc_gh<true, false>), grid, dim3(64), 0, st, g, quad, npts, freqs, l0, m, row0, UG, UH, ld,
                           lstride);
    else if (UH)
        hipLaunchKernelGGL((k_colloc_gh<false, true>), grid, dim3(64), 0, st, g, quad, npts, freqs, l0, m, row0, UG, UH, ld,
                           lstride);
    return hipGetLastError();
}


// Rows per block of the patch kernel: enough to hide a row's start and write-out behind the next one's evaluation and to
// even out chunk counts that are no multiple of 4, and still at least 8192 blocks (16 for each that is resident on 256 CUs)
// where there are as many tiles.
int patch_rows_per_tile(long long tiles) { return (int)std::min<long long>(16, std::max<long long>(1, tiles / 8192)); }

hipError_t launch_colloc_gh_patch(const Geom &g, const double4 *pts, int npts, const Freq *freqs, int l0, int nl, bool real_ends, const Mat &m,
                                 int row0, int nrows, const double4 *tpts, const int *patch_chunk, const int4 *chunk_info,
                                 const int4 *chunk_faces, const int *patch_verts, int npatches, cd *UG, cd *UH, long long ld,
                                 long long lstride, hipStream_t st, const Bands &bands) {
    if ((!UG && !UH) || npts <= 0 || nrows <= 0 || nrows > 65535) return hipErrorInvalidValue;
    if (bands.far_pts && (tpts || bands.far_npts <= 0 || !bands.sphere)) return hipErrorInvalidValue;
    const int slots = real_ends ? std::max(nl - 1, 1) : nl, real_hi = real_ends ? nl - 1 : -1;
    const int rpt = patch_rows_per_tile((long long)npatches * slots * nrows);
    dim3 grid(npatches, slots, (nrows + rpt - 1) / rpt);
#define CQBEM_PATCH(DG, DH, GAL, BANDED)                                                                                    \
    hipLaunchKernelGGL((k_colloc_gh_patch<DG, DH, GAL, BANDED>), grid, dim3(kPatchThreads), 0, st, g, pts, npts, freqs, \
                       l0, m, row0, tpts, patch_chunk, chunk_info, chunk_faces, patch_verts, UG, UH, ld, lstride, nrows, rpt, real_hi, bands)
    if (tpts) {  // test points: never banded (refused above)
        if (UG && UH) CQBEM_PATCH(true, true, true, false);
        else if (UG) CQBEM_PATCH(true, false, true, false);
        else CQBEM_PATCH(false, true, true, false);
    } else if (bands.far_pts) {
        if (UG && UH) CQBEM_PATCH(true, true, false, true);
        else if (UG) CQBEM_PATCH(true, false, false, true);
        else CQBEM_PATCH(false, true, false, true);
    } else {
        if (UG && UH) CQBEM_PATCH(true, true, false, false);
        else if (UG) CQBEM_PATCH(true, false, false, false);
        else CQBEM_PATCH(false, true, false, false);
    }
#undef CQBEM_PATCH
    return hipGetLastError();
}
hipError_t launch_scene_gh(const ScenePiece *pieces, int npieces, long long ntiles, unsigned *counter, bool G, bool H,
                                int num_cus, hipStream_t st) {
    if ((!G && !H) || npieces <= 0 || ntiles <= 0 || ntiles >= (1LL << 31)) return hipErrorInvalidValue;
    const char *env = std::getenv("CQBEM_SCENE_KERNEL");  // read per launch (tests switch it)
    const bool persistent = env && !std::strcmp(env, "persistent");
    if (!persistent) {
        // a dispatch holds fewer than 2^32 work-items: grids of at most 2^22 blocks of 256, in tile order
        constexpr long long kChunk = 1LL << 22;
        for (long long t0 = 0; t0 < ntiles; t0 += kChunk) {
            const dim3 grid((unsigned)std::min(kChunk, ntiles - t0));
            if (G && H)
                hipLaunchKernelGGL((k_scene_gh_tiles<true, true>), grid, dim3(kPatchThreads), 0, st, pieces, npieces, (unsigned)t0);
            else if (G)
                hipLaunchKernelGGL((k_scene_gh_tiles<true, false>), grid, dim3(kPatchThreads), 0, st, pieces, npieces, (unsigned)t0);
            else
                hipLaunchKernelGGL((k_scene_gh_tiles<false, true>), grid, dim3(kPatchThreads), 0, st, pieces, npieces, (unsigned)t0);
        }
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(64), 0, st, counter);
    const unsigned blocks = (unsigned)std::min<long long>(ntiles, 2LL * num_cus);
    if (G && H)
        hipLaunchKernelGGL((k_scene_gh_persistent<true, true>), dim3(blocks), dim3(kPatchThreads), 0, st, pieces, npieces,
                           (unsigned)ntiles, counter);
    else if (G)
        hipLaunchKernelGGL((k_scene_gh_persistent<true, false>), dim3(blocks), dim3(kPatchThreads), 0, st, pieces, npieces,
                           (unsigned)ntiles, counter);
    else
        hipLaunchKernelGGL((k_scene_gh_persistent<false, true>), dim3(blocks), dim3(kPatchThreads), 0, st, pieces, npieces,
                           (unsigned)ntiles, counter);
    return hipGetLastError();
}

int patch_size() { return kPatchVerts; }
int chunk_face_count() { return 64; }

template <bool GAL, bool BANDED>
static hipError_t launch_b(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, bool real_ends,
                           const Mat &m, int row0, int nrows, const double4 *tpts, cd *Bt, cd *Ba, long long out_rows,
                           hipStream_t st, const FaceBands &fb) {
    const int slots = real_ends ? std::max(nl - 1, 1) : nl, real_hi = real_ends ? nl - 1 : -1;
    hipLaunchKernelGGL((k_colloc_b<GAL, BANDED>), dim3(slots, nrows), dim3(256), 0, st, g, quad, npts, freqs, l0, m, row0, tpts, Bt,
                       Ba, out_rows, real_hi, fb);
    return hipGetLastError();
}

hipError_t launch_colloc_b(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, bool real_ends, const Mat &m,
                           int row0, int nrows, cd *Bt, cd *Ba, hipStream_t st, const FaceBands &fb) {
    if (nrows <= 0 || nrows > 65535) return hipErrorInvalidValue;
    return fb.sphere ? launch_b<false, true>(g, quad, npts, freqs, l0, nl, real_ends, m, row0, nrows, nullptr, Bt, Ba, 3LL * g.nv, st, fb)
                     : launch_b<false, false>(g, quad, npts, freqs, l0, nl, real_ends, m, row0, nrows, nullptr, Bt, Ba, 3LL * g.nv, st, fb);
}

hipError_t launch_points_b(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, bool real_ends, const Mat &m,
                           const double4 *tpts, int row0, int nrows, cd *Bt, cd *Ba, long long out_rows, hipStream_t st) {
    if (nrows <= 0 || nrows > 65535 || 3LL * nrows > out_rows) return hipErrorInvalidValue;
    return launch_b<true, false>(g, quad, npts, freqs, l0, nl, real_ends, m, row0, nrows, tpts, Bt, Ba, out_rows, st, FaceBands{});
}

hipError_t launch_colloc_singular(int kind, const Geom &g, const double2 *line, int nline, const Freq *freqs, int l0, int nl,
                                  const Mat &m, int row0, int nrows, cd *U, long long ld, long long lstride, cd *Bt,
                                  cd *Ba, hipStream_t st) {
    const long long n = (long long)nrows * nl;
    if (n <= 0 || n > 0x7fffffffLL) return hipErrorInvalidValue;
    dim3 grid((unsigned)n);  // one wavefront per (row, frequency)
    if (kind == 0)
        hipLaunchKernelGGL((k_colloc_singular<0>), grid, dim3(64), 0, st, g, line, nline, freqs, l0, nl, m, row0, nrows, U,
                           ld, lstride, Bt, Ba, 3LL * g.nv);
    else if (kind == 1)
        hipLaunchKernelGGL((k_colloc_singular<1>), grid, dim3(64), 0, st, g, line, nline, freqs, l0, nl, m, row0, nrows, U,
                           ld, lstride, Bt, Ba, 3LL * g.nv);
    else
        hipLaunchKernelGGL((k_colloc_singular<2>), grid, dim3(64), 0, st, g, line, nline, freqs, l0, nl, m, row0, nrows, U,
                           ld, lstride, Bt, Ba, 3LL * g.nv);
    return hipGetLastError();
}

template <class OutT>
static hipError_t launch_transform_t(const cd *spec, long long E, long long spec_ls, int Lf, const double2 *tab, int L,
                                     OutT *out, long long out_nstride, int num_cus, hipStream_t st) {
    // two entries per lane.  Where the pairs' stores are not aligned (odd sizes or strides, an output at an odd value) they
    // are declared so; one entry per lane with stores of one value took 2.0 ms where this takes 1.64 (3291 x 3291, L = 21, G and H)
    if (Lf <= kTransformMaxLf) {
        const bool aligned = E % 2 == 0 && out_nstride % 2 == 0 && reinterpret_cast<uintptr_t>(out) % (2 * sizeof(OutT)) == 0;
        const long long pblocks = ((E + 1) / 2 + 255) / 256;
        for (int n0 = 0; n0 < L; n0 += kTransformNC) {
            if (aligned)
                hipLaunchKernelGGL((k_transform_pair<2, true, OutT>), dim3((unsigned)pblocks), dim3(256), 0, st, spec, E, spec_ls,
                                   Lf, tab, L, n0, out, out_nstride);
            else
                hipLaunchKernelGGL((k_transform_pair<2, false, OutT>), dim3((unsigned)pblocks), dim3(256), 0, st, spec, E, spec_ls,
                                   Lf, tab, L, n0, out, out_nstride);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    long long blocks = (E + 255) / 256;
    const long long cap = (long long)num_cus * 64;
    if (blocks > cap) blocks = cap;
    if (blocks < 1) blocks = 1;
    for (int n0 = 0; n0 < L; n0 += kTransformNC) {
        hipLaunchKernelGGL((k_transform_wide<kTransformNC, OutT>), dim3((unsigned)blocks), dim3(256), 0, st, spec, E, spec_ls, Lf,
                           tab, L, n0, out, out_nstride);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}
hipError_t launch_transform(const cd *spec, long long E, long long spec_ls, int Lf, const double2 *tab, int L, double *out,
                            long long out_nstride, int num_cus, hipStream_t st) {
    return launch_transform_t(spec, E, spec_ls, Lf, tab, L, out, out_nstride, num_cus, st);
}
hipError_t launch_transform(const cd *spec, long long E, long long spec_ls, int Lf, const double2 *tab, int L, float *out,
                            long long out_nstride, int num_cus, hipStream_t st) {
    return launch_transform_t(spec, E, spec_ls, Lf, tab, L, out, out_nstride, num_cus, st);
}

// CQBEM_HISTORY_ROWS = 1 selects the 8-byte one-row history and matvec kernel, 2 or 4 that many rows per wavefront of the
// 16-byte one, unsplit; anything else (0) the rule below.  Read at every call (a few hundred ns against a launch).
static int history_rows() {
    const char *e = std::getenv("CQBEM_HISTORY_ROWS");
    const int v = e ? std::atoi(e) : 0;
    return v == 1 || v == 2 || v == 4 ? v : 0;
}

// How the rows and the m steps (m = 1: a matvec) go over the wavefronts.  What counts below some 2000 wavefronts is how
// many loads are in flight, beyond that how often the vectors are read again.  us per call, with 4 rows per wavefront and
// no split first: n3 = 486, 31 steps 36 -> 10; 1158, 16 steps 34 -> 20 (22 at 4 rows); 1926, 16 steps 63 -> 42 (45 at
// 2 rows); 7686, 31 steps 4660 and 4650.  One step: 1926 rows 19.7 -> 18.0 at one row, 3489 30.5 at 4 and 29.3 at 2,
// 7686 89.7 at 4 and 95.4 at one.
struct HistorySplit {
    int rows;    // rows per wavefront; 0: the 8-byte kernel
    bool split;  // a block's 4 waves share its rows and take every fourth step each
};
static HistorySplit history_split(long long n3, int m, bool a16) {
    if (const int forced = history_rows()) return {forced == 1 ? 0 : forced, false};
    // unaligned 16-byte loads pay from 4 steps or 2048 rows on (903 rows, 2 steps: 18.3 us in 8-byte loads, 19.4), for one
    // step from 8192 (5001 rows: 40 and 47 us; 12289: 257 and 194).  That is for weights that come from memory (1503 rows,
    // 5 steps: 95 and 60 us; 2601, 2 steps: 101 and 62); the same few steps repeated on weights that the 256 MB cache
    // still holds are up to 1.15 times faster in 8-byte loads (51 and 57; 50 and 58)
    if (m > 1 && (a16 || m >= 4 || n3 >= 2048)) {
        // idle share of 256 CUs in the last round of blocks: 2 rows where that is clearly the smaller one (3489 rows, 16
        // steps, unaligned: 528 us at 2 and 543 at 4 rows; 903: 57 and 53)
        auto uneven = [&](long long r) {
            const long long blocks = (n3 + r - 1) / r;
            return (double)((blocks + 255) / 256) * 256 / (double)blocks;
        };
        return {uneven(4) > 1.06 * uneven(2) ? 2 : 4, true};
    }
    if (!a16 && n3 < 8192) return {0, false};
    return {n3 < 3072 ? 1 : n3 < 6144 ? 2 : 4, false};
}

template <int R, bool A16, bool SPLIT, class S>
static void launch_history_r(const S *G, const S *H, const double *B, const double *p, const double *u,
                              const double *acc, long long n3, long long mat_stride, int m, int nh, double *b,
                              hipStream_t st) {
    const long long waves = (n3 + R - 1) / R;
    const dim3 grid((unsigned)(SPLIT ? waves : (waves + 3) / 4));
    if (G && H)
        hipLaunchKernelGGL((k_history_v2<S, A16, SPLIT, true, true, R>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, mat_stride, m,
                           nh, b);
    else if (G)
        hipLaunchKernelGGL((k_history_v2<S, A16, SPLIT, true, false, R>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, mat_stride, m,
                           nh, b);
    else if (H)
        hipLaunchKernelGGL((k_history_v2<S, A16, SPLIT, false, true, R>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, mat_stride, m,
                           nh, b);
    else
        hipLaunchKernelGGL((k_history_v2<S, A16, SPLIT, false, false, R>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, mat_stride,
                           m, nh, b);
}

template <bool A16, class S>
static void launch_history_v2(HistorySplit h, const S *G, const S *H, const double *B, const double *p, const double *u,
                              const double *acc, long long n3, long long mat_stride, int m, int nh, double *b, hipStream_t st) {
    auto go = [&](auto rows, auto split) {
        launch_history_r<decltype(rows)::value, A16, decltype(split)::value>(G, H, B, p, u, acc, n3, mat_stride, m, nh, b, st);
    };
    using std::integral_constant;
    if (h.split) {
        if (h.rows == 4) go(integral_constant<int, 4>{}, std::true_type{});
        else go(integral_constant<int, 2>{}, std::true_type{});
    } else {
        if (h.rows == 4) go(integral_constant<int, 4>{}, std::false_type{});
        else if (h.rows == 2) go(integral_constant<int, 2>{}, std::false_type{});
        else go(integral_constant<int, 1>{}, std::false_type{});
    }
}

static bool aligned16(const double *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }
static bool aligned8(const void *q) { return (reinterpret_cast<uintptr_t>(q) & 7) == 0; }

hipError_t launch_history_f32(const float *G, const float *H, const double *B, const double *p, const double *u,
                              const double *acc, long long n3, int m, int nh, double *b, hipStream_t st) {
    // single-precision matrices: 8-byte pairs of weights against 16-byte pairs of history entries
    if (n3 % 2 != 0 || (G && (!aligned8(G) || !aligned16(p))) || (H && (!aligned8(H) || !aligned16(u))))
        return hipErrorInvalidValue;
    HistorySplit h = history_split(n3, m, true);
    if (h.rows == 0) h.rows = 4;  // there is no kernel of single loads
    launch_history_v2<true>(h, G, H, B, p, u, acc, n3, n3 * n3, m, nh, b, st);
    return hipGetLastError();
}

hipError_t launch_history(const double *G, const double *H, const double *B, const double *p, const double *u,
                          const double *acc, long long n3, int m, int nh, double *b, hipStream_t st) {
    const bool a16 = n3 % 2 == 0 && (!G || (aligned16(G) && aligned16(p))) && (!H || (aligned16(H) && aligned16(u)));
    const bool a8 = (!G || (aligned8(G) && aligned8(p))) && (!H || (aligned8(H) && aligned8(u)));
    const HistorySplit h = history_split(n3, m, a16);
    if (h.rows && a8) {
        if (a16) launch_history_v2<true>(h, G, H, B, p, u, acc, n3, n3 * n3, m, nh, b, st);
        else launch_history_v2<false>(h, G, H, B, p, u, acc, n3, n3 * n3, m, nh, b, st);
        return hipGetLastError();
    }
    const dim3 grid((unsigned)((n3 + 3) / 4));
    if (G && H)
        hipLaunchKernelGGL((k_history<true, true>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, m, nh, b);
    else if (G)
        hipLaunchKernelGGL((k_history<true, false>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, m, nh, b);
    else if (H)
        hipLaunchKernelGGL((k_history<false, true>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, m, nh, b);
    else
        hipLaunchKernelGGL((k_history<false, false>), grid, dim3(256), 0, st, G, H, B, p, u, acc, n3, m, nh, b);
    return hipGetLastError();
}

hipError_t launch_matvec(const double *A, const double *x, long long n, double *y, hipStream_t st) {
    const bool a16 = n % 2 == 0 && aligned16(A) && aligned16(x);
    const HistorySplit h = history_split(n, 1, a16);
    if (h.rows && aligned8(A) && aligned8(x)) {
        if (a16) launch_history_v2<true, double>(h, A, nullptr, nullptr, x, nullptr, nullptr, n, 0, 1, 1, y, st);
        else launch_history_v2<false, double>(h, A, nullptr, nullptr, x, nullptr, nullptr, n, 0, 1, 1, y, st);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_matvec, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st, A, x, n, y);
    return hipGetLastError();
}

hipError_t launch_add_c_colloc(double *H0, const double *C, int nv, hipStream_t st) {
    hipLaunchKernelGGL(k_add_c_colloc<double>, dim3((9 * nv + 255) / 256), dim3(256), 0, st, H0, C, nv);
    return hipGetLastError();
}
hipError_t launch_add_c_colloc(float *H0, const double *C, int nv, hipStream_t st) {
    hipLaunchKernelGGL(k_add_c_colloc<float>, dim3((9 * nv + 255) / 256), dim3(256), 0, st, H0, C, nv);
    return hipGetLastError();
}

hipError_t launch_add_triplets(double *H0, const long long *idx, const double *val, long long n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_add_triplets<double>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, H0, idx, val, n);
    return hipGetLastError();
}
hipError_t launch_add_triplets(float *H0, const long long *idx, const double *val, long long n, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_add_triplets<float>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, H0, idx, val, n);
    return hipGetLastError();
}

hipError_t launch_b_post(double *Bt, double *Ba, double *B6, const double *V, int nv, int L, hipStream_t st) {
    const long long n = 3LL * nv * L;
    hipLaunchKernelGGL(k_b_post, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, Bt, Ba, B6, V, nv, L);
    return hipGetLastError();
}

}  // namespace cqbem
