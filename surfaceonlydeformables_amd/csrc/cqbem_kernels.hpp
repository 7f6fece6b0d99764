// Kernel-side data structures and launchers shared by the host driver.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "cqbem_device.hpp"

namespace cqbem {

// Device-resident mesh of one job.
struct Geom {
    const double *V;     // nv x 3
    const int *F;        // nf x 3
    const double *N;     // nf x 3 unit normals
    const double *area;  // nf
    const int *vs_ptr;   // nv+1: vertex star CSR (faces incident to each vertex)
    const int *vs_face;  // (face << 2) | corner, ascending face index
    const int *sg_ptr;   // nv+1: faces singular for each collocation vertex
    const int *sg_face;  // (face << 2) | first matching corner
    const int *vmap;     // nullable vertex_map_inverse
    int nv, nf;
};

hipError_t launch_colloc_gh(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, const Mat &m,
                            int row0, int nrows, cd *UG, cd *UH, long long ld, long long lstride, hipStream_t st);

// Distance bands of the patch kernel's regular-face rule (CQBEM_QUAD_BANDED).  A tile (patch, row point x) takes the
// far rule at every frequency when |x - centre| >= radius + kappa h (h: the patch's largest face diameter);
// otherwise the reference rule.  far_pts == nullptr: the reference rule for every tile.
struct Bands {
    const double4 *far_pts = nullptr;  // patch point table of the far rule (layout of the reference rule's)
    int far_npts = 0;
    const double4 *sphere = nullptr;   // per patch: centre, radius + kappa h
};
// The bands' rule choice: whether row point x lies at or beyond distance S.w from (S.x, S.y, S.z).  Compiled without
// contraction, so that the host plans and the kernels decide every tile and face alike.
__host__ __device__ inline bool beyond_sphere(double x0, double x1, double x2, const double4 &S) {
#pragma clang fp contract(off)
    const double dx = x0 - S.x, dy = x1 - S.y, dz = x2 - S.z;
    return dx * dx + dy * dy + dz * dz >= S.w * S.w;
}
// Of the waves that share a chunk of the patch kernel, wave `part` takes the rule's points from `part` on.  A far rule may
// have fewer points than the waves that the reference rule calls for: the last ones then have none.
__host__ __device__ inline bool part_has_points(int npts, int part) { return part < npts; }
// The points that it takes, every split-th one; the first is told apart (it starts the sums).  part_has_points.
template <class Point> __host__ __device__ __attribute__((always_inline)) inline void each_part_point(int npts, int split, int part, const Point &point) {
    point(part, std::true_type{});
#pragma unroll 1
    for (int q = part + split; q < npts; q += split) point(q, std::false_type{});
}
// The update of every lane whose sub-step is `step`, the sub-steps one after another: sync() orders the lanes of the wave,
// so that an update sees those of the sub-steps before it, whichever lanes made them.
template <class Sync, class Update>
__host__ __device__ __attribute__((always_inline)) inline void in_sub_steps(int nsub, int step, const Sync &sync, const Update &update) {
    for (int s = 0; s < nsub; ++s) {
        sync();
        if (step == s) update();
    }
}
// Distance bands of the B kernels' regular-face rule (CQBEM_QUAD_BANDED).  Face f takes the far rule for row point x
// at every frequency when |x - centre_f| >= radius_f + kappa h_f (h_f: its longest edge); otherwise the reference
// rule.  sphere == nullptr: the reference rule for every face.
struct FaceBands {
    const double4 *far_quad = nullptr;  // the far rule, (b0, b1, b2, w) per point
    int far_npts = 0;
    const double4 *sphere = nullptr;    // per face: centre, radius + kappa h
};
// Patch form of the G/H regular-face kernel (both matrices): per patch a range of chunks
// [patch_chunk[p], patch_chunk[p+1]) of up to 64 faces; per chunk (first face entry, nfaces, sub-steps of corner 0 |
// of corner 1 << 8 | of corner 2 << 16, 0); per face entry, for its corners k = 0..2 (the face's, from any of the
// three), x, y, z = vertex | slot << 24 and w = the sub-steps, 8 bits each (255: outside the patch).
// `pts` holds, for each point of the rule, (b1, b2, 0, 0) and w (b0, b1, b2, 1).
// real_ends: s is real at the first and the last of the nl frequencies (the half spectrum of an even L, or one real
// frequency), which then share one slot of the grid.
// Rows are collocation vertices row0..row0+nrows-1 when tpts is null.  Otherwise they are the test points
// tpts[row0..row0+nrows-1] = (x, y, z, test face), each excluding every face that shares a vertex with its
// test face (the Galerkin non-singular set), and row r of the launch goes to rows 3r..3r+2 of UG/UH.
hipError_t launch_colloc_gh_patch(const Geom &g, const double4 *pts, int npts, const Freq *freqs, int l0, int nl, bool real_ends,
                                 const Mat &m,
                                 int row0, int nrows, const double4 *tpts, const int *patch_chunk, const int4 *chunk_info,
                                 const int4 *chunk_faces, const int *patch_verts, int npatches, cd *UG, cd *UH, long long ld,
                                 long long lstride, hipStream_t st, const Bands &bands = Bands{});
int patch_size();       // vertex slots per patch
int chunk_face_count();  // faces per chunk
int patch_rows_per_tile(long long tiles);  // rows per block for a job of `tiles` (patch, frequency, row) tiles

// One object's row slab in a multi-object launch of the patch kernel (collocation rows row0..row0+nrows-1 at all
// nl frequencies of `freqs`): its npatches x slots x ceil(nrows / rpt) tiles of rpt rows are numbered from base; slots: nl, or nl - 1 with
// real_hi = nl - 1 when the first and the last frequency share one).
struct ScenePiece {
    Geom g;
    const double4 *pts;
    int npts;
    const Freq *freqs;
    Mat m;
    int row0, nrows, rpt, slots, real_hi, npatches;
    const int *patch_chunk;
    const int4 *chunk_info;
    const int4 *chunk_faces;
    const int *patch_verts;
    cd *UG, *UH;
    long long ld, lstride;
    unsigned base;
    Bands bands;
};
// The pieces (device array, ascending base, all with the same G / H selection): one block per tile, or with
// CQBEM_SCENE_KERNEL=persistent min(ntiles, 2 per CU) blocks that take tiles from *counter (zeroed by the launcher with a
// kernel).
hipError_t launch_scene_gh(const ScenePiece *pieces, int npieces, long long ntiles, unsigned *counter, bool G, bool H,
                                int num_cus, hipStream_t st);
hipError_t launch_colloc_b(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, bool real_ends,
                                 const Mat &m,
                           int row0, int nrows, cd *Bt, cd *Ba, hipStream_t st, const FaceBands &fb = FaceBands{});
// B_trans / B_angular rows of the test points tpts[row0..row0+nrows-1] (Galerkin non-singular set, as above), into
// rows 3r..3r+2 of Bt (out_rows x 3 per frequency) and Ba (out_rows x 9).
hipError_t launch_points_b(const Geom &g, const double4 *quad, int npts, const Freq *freqs, int l0, int nl, bool real_ends,
                                 const Mat &m,
                           const double4 *tpts, int row0, int nrows, cd *Bt, cd *Ba, long long out_rows, hipStream_t st);
hipError_t launch_colloc_singular(int kind, const Geom &g, const double2 *line, int nline, const Freq *freqs, int l0, int nl,
                                  const Mat &m, int row0, int nrows, cd *U, long long ld, long long lstride, cd *Bt,
                                  cd *Ba, hipStream_t st);
// out[n * out_nstride + e] = sum_l Re(spec[l * spec_ls + e] T(n, l)) for e < E (spec_ls >= E: a slab buffer may be
// sized for more rows than the slab holds).
hipError_t launch_transform(const cd *spec, long long E, long long spec_ls, int Lf, const double2 *tab, int L, double *out,
                            long long out_nstride,
                            int num_cus, hipStream_t st);
// The same with the weights rounded to float (resident storage in single precision).
hipError_t launch_transform(const cd *spec, long long E, long long spec_ls, int Lf, const double2 *tab, int L, float *out,
                            long long out_nstride, int num_cus, hipStream_t st);
hipError_t launch_add_c_colloc(double *H0, const double *C, int nv, hipStream_t st);
hipError_t launch_add_c_colloc(float *H0, const double *C, int nv, hipStream_t st);
// b = sum_{i=1..m} (G_i p[nh-i] - H_i u[nh-i] + B_i acc[nh-i]); any of G, H, B may be null.
hipError_t launch_history(const double *G, const double *H, const double *B, const double *p, const double *u,
                          const double *acc, long long n3, int m, int nh, double *b, hipStream_t st);
hipError_t launch_matvec(const double *A, const double *x, long long n, double *y, hipStream_t st);
hipError_t launch_add_triplets(double *H0, const long long *idx, const double *val, long long n, hipStream_t st);
hipError_t launch_add_triplets(float *H0, const long long *idx, const double *val, long long n, hipStream_t st);
// The history sum with G_i, H_i stored in float (n3 even, G/H 8-byte and p/u 16-byte aligned).
hipError_t launch_history_f32(const float *G, const float *H, const double *B, const double *p, const double *u,
                              const double *acc, long long n3, int m, int nh, double *b, hipStream_t st);
hipError_t launch_b_post(double *Bt, double *Ba, double *B6, const double *V, int nv, int L, hipStream_t st);

}  // namespace cqbem
