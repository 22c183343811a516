// HIP kernels of the gfx950 rasterizer.
//
// Pipeline for a batch of views (a single view is a batch of one):
//   k_face_soup   48-byte face records (positions, face normal) per mesh
//   k_begin       view descriptors, per-tile bin counters and status words
//   k_setup_bin   per-face setup of the face loop (rasterizer.cc:162-193):
//                 z<0 reject, bbox, off-screen cull, pixel bbox, area; then
//                 appends (face id, skip depth) to the front or back segment
//                 of every screen tile its pixel bbox touches (a face of at
//                 most 4 bbox pixels only where it may cover a pixel centre)
//   k_raster      one workgroup per screen tile: stages the tile's faces in
//                 LDS (skipping faces proven hidden), expands (face, pixel)
//                 pairs so every lane tests one pair, resolves depth with a
//                 packed 64-bit (depth bits << 32 | face id) LDS atomicMin,
//                 then shades and writes every output pixel of the tile once
//                 (resolve loop rasterizer.cc:243-301, pixel_shader.h).
//
// Bit-exactness: all coverage arithmetic follows the reference's expression
// order; this file is compiled with -ffp-contract=off and correctly rounded
// fp32 division/sqrt (see the Makefile), and the pragma below forbids
// contraction locally as well.

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <float.h>
#include <limits.h>

#include "binning.h"
#include "device_common.h"

#pragma clang fp contract(off)

namespace ugu_hip {

// w2c_R * p + w2c_t, then PinholeCamera::Project (camera.h:380-387):
// x = fx / z * x + cx (divide first), y likewise, z kept.
UGU_DEV float4 project_point(const DevView& v, float px, float py, float pz) {
  float qx = sum3(v.w2c_R[0] * px, v.w2c_R[1] * py, v.w2c_R[2] * pz) + v.w2c_t[0];
  float qy = sum3(v.w2c_R[3] * px, v.w2c_R[4] * py, v.w2c_R[5] * pz) + v.w2c_t[1];
  float qz = sum3(v.w2c_R[6] * px, v.w2c_R[7] * py, v.w2c_R[8] * pz) + v.w2c_t[2];
  // fx / qz and fy / qz are the same correctly rounded quotient when fx == fy
  // (a wave-uniform branch: the second divide is not executed then)
  const float sx = v.fx / qz;
  float sy = sx;
  if (__builtin_expect(v.fy != v.fx, 0)) sy = v.fy / qz;
  float4 r;
  r.x = sx * qx + v.cx;
  r.y = sy * qy + v.cy;
  r.z = qz;
  r.w = 0.0f;
  return r;
}

// A face record is three float4: (x0 y0 z0 x1) (y1 z1 x2 y2) (z2 nx ny nz),
// the face's vertex positions and its face normal.
UGU_DEV void load_face_rec(const float4* soup, int f, float P[9], float N[3]) {
  const float4* r = soup + int64_t(f) * 3;
  const float4 a = r[0], b = r[1], c = r[2];
  P[0] = a.x; P[1] = a.y; P[2] = a.z;
  P[3] = a.w; P[4] = b.x; P[5] = b.y;
  P[6] = b.z; P[7] = b.w; P[8] = c.x;
  N[0] = c.y; N[1] = c.z; N[2] = c.w;
}

// True when the screen x, y of the three corners are all below 2^30 in
// magnitude (no NaN or infinity): the sum of their magnitudes propagates NaN
// and exceeds 2^30 whenever one of them does.
UGU_DEV bool small_screen(const float4& a, const float4& b, const float4& c) {
  return ((fabsf(a.x) + fabsf(b.x)) + (fabsf(c.x) + fabsf(a.y))) + (fabsf(b.y) + fabsf(c.y)) <
         1073741824.0f;
}

// Per-face setup of rasterizer.cc:164-193. Returns false when the
// reference skips the face or its pixel bbox is empty.
UGU_DEV bool face_setup(const float4& a, const float4& b, const float4& c,
                        int W, int H, int& x0, int& x1, int& y0, int& y1,
                        float& area) {
  if (a.z < 0.0f || b.z < 0.0f || c.z < 0.0f) return false;
  if (small_screen(a, b, c)) {
    // no NaN: std::min / std::max are the hardware min / max (their choice
    // between +0 and -0 aside, which ceil, floor and the comparisons below
    // do not see), and below 2^30 the x86 conversions are plain truncations
    const float xmin = fminf(fminf(a.x, b.x), c.x), xmax = fmaxf(fmaxf(a.x, b.x), c.x);
    const float ymin = fminf(fminf(a.y, b.y), c.y), ymax = fmaxf(fmaxf(a.y, b.y), c.y);
    if (xmin > static_cast<float>(W - 1) || xmax < 0.0f ||
        ymin > static_cast<float>(H - 1) || ymax < 0.0f)
      return false;
    x0 = max(0, static_cast<int>(ceilf(xmin)));
    x1 = min(W - 1, static_cast<int>(floorf(xmax)));
    y0 = max(0, static_cast<int>(ceilf(ymin)));
    y1 = min(H - 1, static_cast<int>(floorf(ymax)));
    area = edge_fn(a.x, a.y, b.x, b.y, c.x, c.y);
    if (fabsf(area) < FLT_MIN) return false;
    return x0 <= x1 && y0 <= y1;
  }
  float xmin = min3_std(a.x, b.x, c.x);
  float ymin = min3_std(a.y, b.y, c.y);
  float xmax = max3_std(a.x, b.x, c.x);
  float ymax = max3_std(a.y, b.y, c.y);
  if (xmin > static_cast<float>(W - 1) || xmax < 0.0f ||
      ymin > static_cast<float>(H - 1) || ymax < 0.0f)
    return false;
  x0 = max(0, f2i_x86(ceilf(xmin)));
  x1 = min(W - 1, f2i_sat(floorf(xmax)));
  y0 = max(0, f2i_x86(ceilf(ymin)));
  y1 = min(H - 1, f2i_sat(floorf(ymax)));
  area = edge_fn(a.x, a.y, b.x, b.y, c.x, c.y);
  if (fabsf(area) < FLT_MIN) return false;
  return x0 <= x1 && y0 <= y1;
}

// Coverage, perspective-correct weights and depth of one (face, pixel) pair
// (rasterizer.cc:196-226). Returns true when the pixel is covered.
UGU_DEV bool cover_test(float ax, float ay, float az, float bx, float by,
                        float bz, float cx, float cy, float cz, float area,
                        bool bf, float x, float y, float& z, float& w0o,
                        float& w1o, float& w2o) {
  float w0 = edge_fn(bx, by, cx, cy, x, y);
  float w1 = edge_fn(cx, cy, ax, ay, x, y);
  float w2 = edge_fn(ax, ay, bx, by, x, y);
  bool cov = (!bf && (w0 >= 0.0f && w1 >= 0.0f && w2 >= 0.0f)) ||
             (bf && (w0 <= 0.0f && w1 <= 0.0f && w2 <= 0.0f));
  if (!cov) return false;
  w0 /= area;
  w1 /= area;
  w2 /= area;
  w0 /= az;
  w1 /= bz;
  w2 /= cz;
  z = 1.0f / (w0 + w1 + w2);
  w0o = w0 * z;
  w1o = w1 * z;
  w2o = w2 * z;
  return true;
}



// ---------------------------------------------------------------------------
// k_begin

// Starts a pass: clears the tiles' counters and the status words and, with
// N > 0, writes the view descriptors it got as arguments to device memory (one
// launch in place of a host copy and a clear: the copy's start and the wait
// between it and the next kernel cost more than either).
// Four words per tile: front and back segment counters, the minimum skip depth
// of the back segment (bits; +inf) and the tile's view (largest v with
// views[v].tile_base <= tile), so the tile kernels read their counters and find
// their view with one load. The tile kernels put the first three words back, so
// a pass of one view (view word 0) needs no clearing when the counters it uses
// were left by such passes: its setup kernel takes the descriptor and clears the
// status. 32 k faces at 640x480: 93 us with two copies, a clear and a status
// copy around setup and raster, 75 us with this kernel and the status in a
// pinned word, 69 us without it.
template <int N>
__global__ __launch_bounds__(256) void k_begin(InlineViews<N == 0 ? 1 : N> arg,
                                               const DevView* __restrict__ views, DevView* out,
                                               int32_t n_views, int32_t* counts, int32_t n_tiles,
                                               int32_t* status) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_tiles) {
    int view = 0;
    if (N > 0) {
#pragma unroll
      for (int k = 1; k < N; k++) view = (k < n_views && arg.v[k].tile_base <= i) ? k : view;
    } else {
      int hi = n_views - 1;
      while (view < hi) {
        const int mid = (view + hi + 1) >> 1;
        if (views[mid].tile_base <= i) view = mid; else hi = mid - 1;
      }
    }
    reinterpret_cast<int4*>(counts)[i] = make_int4(0, 0, 0x7f800000, view);
  }
  if (blockIdx.x == 0) {
    if (status) clear_status(status);
    if (N > 0) store_inline_views(out, n_views);
  }
}

// ---------------------------------------------------------------------------
// Mesh::CalcFaceNormal (src/mesh.cc:339-349) pieces, for the differentiable
// path where positions change between calls.

UGU_DEV void normalize3(float& x, float& y, float& z) {
  float n = sum3(x * x, y * y, z * z);
  if (n > 0.0f) {
    float s = sqrtf(n);
    x = x / s;
    y = y / s;
    z = z / s;
  }
}


// ---------------------------------------------------------------------------
// k_shade_rec: one 64-byte shading record per face (DevMesh::shade): the
// corners' uvs (uv[uv_indices]), the material id and the corners' vertex
// normals (normals[normal_indices]), copied bit for bit (zero where the mesh
// has none), so the resolve fetches a winner's shading inputs with one load.
// Layout (u0 v0 u1 v1)(u2 v2 mat n0x)(n0y n0z n1x n1y)(n1z n2x n2y n2z): the
// texture inputs are the first 32 bytes, the normals the last 36.
__global__ void k_shade_rec(DevMesh m, float4* __restrict__ out) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= m.F) return;
  float u[6] = {0, 0, 0, 0, 0, 0}, n[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  if (m.uv && m.uvidx)
    for (int k = 0; k < 3; k++) {
      const float* q = m.uv + int64_t(m.uvidx[int64_t(f) * 3 + k]) * 2;
      u[2 * k] = q[0];
      u[2 * k + 1] = q[1];
    }
  if (m.normals && m.nidx)
    for (int k = 0; k < 3; k++) {
      const float* q = m.normals + int64_t(m.nidx[int64_t(f) * 3 + k]) * 3;
      n[3 * k] = q[0];
      n[3 * k + 1] = q[1];
      n[3 * k + 2] = q[2];
    }
  const int mat = m.matid ? m.matid[f] : 0;
  float4* r = out + int64_t(f) * 4;
  r[0] = make_float4(u[0], u[1], u[2], u[3]);
  r[1] = make_float4(u[4], u[5], __int_as_float(mat), n[0]);
  r[2] = make_float4(n[1], n[2], n[3], n[4]);
  r[3] = make_float4(n[5], n[6], n[7], n[8]);
}

// ---------------------------------------------------------------------------
// k_face_soup: one 48-byte record per face (three vertex positions, then the
// face normal) so setup and raster fetch a face with one dependent load
// instead of an index load and three vertex gathers. compute_normals:
// Mesh::CalcFaceNormal on device (differentiable path, the positions change
// every call; also written to fn_out); otherwise the mesh's face normals are
// copied (zero when it has none).

__global__ void k_face_soup(const float* __restrict__ verts, const int32_t* __restrict__ faces,
                            const float* __restrict__ fnormals, int32_t F, int compute_normals,
                            float4* __restrict__ soup, float* __restrict__ fn_out) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= F) return;
  const int32_t* fi = faces + int64_t(f) * 3;
  float P[9];
  for (int k = 0; k < 3; k++) {
    const float* q = verts + int64_t(fi[k]) * 3;
    P[k * 3 + 0] = q[0];
    P[k * 3 + 1] = q[1];
    P[k * 3 + 2] = q[2];
  }
  float nx = 0.0f, ny = 0.0f, nz = 0.0f;
  if (compute_normals) {
    float ax = P[3] - P[0], ay = P[4] - P[1], az = P[5] - P[2];
    float bx = P[6] - P[0], by = P[7] - P[1], bz = P[8] - P[2];
    normalize3(ax, ay, az);
    normalize3(bx, by, bz);
    nx = ay * bz - az * by;
    ny = az * bx - ax * bz;
    nz = ax * by - ay * bx;
    normalize3(nx, ny, nz);
    if (fn_out) {
      fn_out[int64_t(f) * 3 + 0] = nx;
      fn_out[int64_t(f) * 3 + 1] = ny;
      fn_out[int64_t(f) * 3 + 2] = nz;
    }
  } else if (fnormals) {
    nx = fnormals[int64_t(f) * 3 + 0];
    ny = fnormals[int64_t(f) * 3 + 1];
    nz = fnormals[int64_t(f) * 3 + 2];
  }
  float4* r = soup + int64_t(f) * 3;
  r[0] = make_float4(P[0], P[1], P[2], P[3]);
  r[1] = make_float4(P[4], P[5], P[6], P[7]);
  r[2] = make_float4(P[8], nx, ny, nz);
}

// ---------------------------------------------------------------------------
// k_setup_bin: one thread per (face, view)

// Skip depth of a face in a view: a lower bound of every depth the coverage
// test (cover_test) can compute for the face at a pixel of its bbox, or -1
// when no useful bound exists. Once every in-view pixel of a tile holds a depth
// d <= dmax, a face whose skip depth exceeds dmax (1 + 2^-8) can neither win a
// pixel nor produce a depth below FLT_MIN, so the rasterizer drops it without
// fetching it.
// Bound: with L the larger bbox extent, rounding moves each edge function by
// at most 8u L^2 (u = 2^-24) and the area by as much, so the normalised
// weights sum to at most 1 + 32u L^2 / |area|; with 2^-9 L^2 <= |area| that is
// 1 + 2^-10, five more roundings cost < 2^-21, and
// z >= min(za, zb, zc) (1 - 2^-10 - 2^-20). NaN or huge values fail every
// comparison and give -1.
UGU_DEV float skip_depth(const float4& a, const float4& b, const float4& c, float area) {
  float ex, ey;
  if (small_screen(a, b, c)) {
    // no NaN: the hardware min / max (see face_setup)
    ex = fmaxf(fmaxf(a.x, b.x), c.x) - fminf(fminf(a.x, b.x), c.x);
    ey = fmaxf(fmaxf(a.y, b.y), c.y) - fminf(fminf(a.y, b.y), c.y);
  } else {
    ex = max3_std(a.x, b.x, c.x) - min3_std(a.x, b.x, c.x);
    ey = max3_std(a.y, b.y, c.y) - min3_std(a.y, b.y, c.y);
  }
  if (!(ex <= 1048576.0f && ey <= 1048576.0f)) return -1.0f;
  const float L = ex > ey ? ex : ey;
  if (!(L * L * 0.001953125f <= fabsf(area))) return -1.0f;
  if (!(a.z > 0.0f && b.z > 0.0f && c.z > 0.0f)) return -1.0f;
  // three positive depths: std::min is the hardware min
  return fminf(fminf(a.z, b.z), c.z);
}

// Tiles of a small face's bbox (at most kCoverProbe pixel centres, so at most
// 2 x 2 tiles) holding a centre the face may cover: bit (tx - tx0) + 2 (ty -
// ty0). The edge functions are the coverage test's (cover_test, same operands
// and order, so the same bits); a centre where they are neither all >= 0 nor
// all <= 0 is covered for neither back-face flag, so the rasterizer's pair
// test would reject the face there whatever the ray. A face with no such
// centre (most sub-pixel faces) gets no bin entry at all.
template <int TW, int TH>
UGU_DEV uint32_t probe_cover(const float4& a, const float4& b, const float4& c, int x0, int x1,
                             int y0, int y1, int tx0, int ty0) {
  static_assert(TW >= kCoverProbe && TH >= kCoverProbe, "a probed bbox spans at most 2 x 2 tiles");
  uint32_t m = 0u;
  int px = x0, py = y0;
#pragma unroll
  for (int k = 0; k < kCoverProbe; k++) {
    if (py <= y1) {
      const float x = static_cast<float>(px), y = static_cast<float>(py);
      const float w0 = edge_fn(b.x, b.y, c.x, c.y, x, y);
      const float w1 = edge_fn(c.x, c.y, a.x, a.y, x, y);
      const float w2 = edge_fn(a.x, a.y, b.x, b.y, x, y);
      // all >= 0 or all <= 0 (a NaN fails both in cover_test; here fminf /
      // fmaxf drop it, which only keeps more centres)
      if (fminf(fminf(w0, w1), w2) >= 0.0f || fmaxf(fmaxf(w0, w1), w2) <= 0.0f)
        m |= 1u << ((static_cast<int>(static_cast<unsigned>(px) / TW) - tx0) +
                    2 * (static_cast<int>(static_cast<unsigned>(py) / TH) - ty0));
      if (++px > x1) {
        px = x0;
        py++;
      }
    }
  }
  return m;
}

// INL: a pass of one view, its descriptor an argument (see k_begin).
template <int TW, int TH, bool INL>
__global__ __launch_bounds__(256) void k_setup_bin(
    InlineViews<1> arg, const DevView* __restrict__ views, DevView* out, int n_views, DevMesh mesh,
    DevBins bins) {
  if (INL && blockIdx.x == 0) {
    clear_status(bins.status);
    store_inline_views(out, 1);
  }
  // The block's 256 faces share their vertices (about 150 distinct ones on a
  // regular mesh): every distinct vertex is projected once per view into LDS
  // and the faces read their corners from there, about 0.6 projections per
  // face instead of three. Without the block lists each face projects its
  // own corners.
  __shared__ float4 sp[768];
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  const bool shared = mesh.blk_off != nullptr;
  int vbase = 0, nu = 0;
  float P[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  int loc[3] = {0, 0, 0};
  if (shared) {
    vbase = mesh.blk_off[blockIdx.x];
    nu = mesh.blk_off[blockIdx.x + 1] - vbase;
    if (f < mesh.F) {
      const uint32_t lc = mesh.face_loc[f];
      loc[0] = lc & 1023u;
      loc[1] = (lc >> 10) & 1023u;
      loc[2] = lc >> 20;
    }
    for (int j = 0; j < 3; j++) {
      const int k = threadIdx.x + j * 256;
      if (k < nu) {
        const float* q = mesh.verts + int64_t(mesh.blk_vid[vbase + k]) * 3;
        P[j * 3 + 0] = q[0];
        P[j * 3 + 1] = q[1];
        P[j * 3 + 2] = q[2];
      }
    }
  } else if (f < mesh.F) {
    float N[3];
    load_face_rec(mesh.soup, f, P, N);
  }
  const int vb = blockIdx.y * kSetupViews;
  const int ve = min(vb + kSetupViews, n_views);
  for (int vi = vb; vi < ve; vi++) {
    const DevView& v = INL ? arg.v[0] : views[vi];
    bool has = false, back = false;
    float zskip = -1.0f;
    int tx0 = 0, tx1 = -1, ty0 = 0, ty1 = -1;
    // tiles of a probed face's bbox that receive it, bit (tx - tx0) + 2 (ty -
    // ty0); all ones for a face that is not probed (every bbox tile)
    uint32_t tmask = ~0u;
    float4 a, b, c;
    if (shared) {
      for (int j = 0; j < 3; j++) {
        const int k = threadIdx.x + j * 256;
        if (k < nu) sp[k] = project_point(v, P[j * 3 + 0], P[j * 3 + 1], P[j * 3 + 2]);
      }
      __syncthreads();
      a = sp[loc[0]];
      b = sp[loc[1]];
      c = sp[loc[2]];
      __syncthreads();  // the next view overwrites the window
    } else {
      a = project_point(v, P[0], P[1], P[2]);
      b = project_point(v, P[3], P[4], P[5]);
      c = project_point(v, P[6], P[7], P[8]);
    }
    if (f < mesh.F) {
      int x0, x1, y0, y1;
      float area;
      if (face_setup(a, b, c, v.W, v.H, x0, x1, y0, y1, area)) {
        has = true;
        // faces that are clockwise on screen are mostly hidden back faces:
        // they go to the back segment so the rasterizer sees them last
        back = !(area > 0.0f);
        zskip = skip_depth(a, b, c, area);
        tx0 = x0 / TW;
        tx1 = x1 / TW;
        ty0 = y0 / TH;
        ty1 = y1 / TH;
        if ((x1 - x0 + 1) * (y1 - y0 + 1) <= kCoverProbe) {
          tmask = probe_cover<TW, TH>(a, b, c, x0, x1, y0, y1, tx0, ty0);
          has = tmask != 0u;
        }
      }
    }
    // one append per tile of the face's pixel bbox (of a probed small face,
    // per tile where it may cover a centre): up to kAppendRounds
    // rounds are issued before any is finished, further rounds (faces over
    // more tiles) one at a time
    const int2 entry = make_int2(f, __float_as_int(zskip));
    // one bound for all rounds: the minimum over every back face of the
    // wavefront is also below the skip depth of each back face of a round
    const uint32_t zmin = back_zmin(has && back, zskip);
    const int nx = tx1 - tx0 + 1;
    const int rest = has ? max(nx * (ty1 - ty0 + 1) - kAppendRounds, 0) : 0;
    int tx = tx0, ty = ty0;
    // a probed face visits only its marked tiles, one per round
    const bool probed = tmask != ~0u;
    uint32_t pm = tmask;
    AppendTicket tk[kAppendRounds];
    int used = 0;  // rounds issued: until no lane has a tile left
#pragma unroll
    for (int r = 0; r < kAppendRounds; r++) {
      if (!__builtin_amdgcn_ballot_w64(has)) break;
      used = r + 1;
      int ax = tx, ay = ty;
      if (probed) {
        const int bit = __ffs(pm) - 1;
        ax = tx0 + (bit & 1);
        ay = ty0 + (bit >> 1);
      }
      const int seg = has ? 4 * (v.tile_base + ay * v.tiles_x + ax) + (back ? 1 : 0) : -1;
      tk[r] = append_issue(bins, seg, zmin, has);
      if (probed) {
        pm &= pm - 1u;
        has = has && pm != 0u;
      } else if (has && ++tx > tx1) {
        tx = tx0;
        if (++ty > ty1) has = false;
      }
    }
    append_finish<kAppendRounds>(bins, tk, &entry, used);
    // Faces over more than kAppendRounds tiles (large triangles): their
    // remaining tiles, all lanes' together, 64 per round -- lane j of a round
    // takes pair base + j of the wavefront's list, finds its face's lane (the
    // last lane whose exclusive prefix is <= the pair) and the tile ordinal.
    if (__any(rest > 0)) {
      const int lane = __lane_id();
      const int incl = wave_incl_sum(rest);
      const int excl = incl - rest;
      const int total = __builtin_amdgcn_readlane(incl, 63);
      for (int base = 0; base < total; base += 64) {
        const int p = base + lane;
        int src = 0;
        for (int step = 32; step >= 1; step >>= 1)
          if (__shfl(excl, src + step) <= p) src += step;
        const int k = p - __shfl(excl, src) + kAppendRounds;
        // lanes past the last pair (act false) may land on a face without
        // tiles (nx 0): clamp so their unused division stays defined
        const int snx = max(__shfl(nx, src), 1);
        const int sty = __shfl(ty0, src) + k / snx;
        const int stx = __shfl(tx0, src) + k % snx;
        const int sback = __shfl(back ? 1 : 0, src);
        const int2 e = make_int2(__shfl(f, src), __shfl(__float_as_int(zskip), src));
        const bool act = p < total;
        const AppendTicket t1 = append_issue(
            bins, act ? 4 * (v.tile_base + sty * v.tiles_x + stx) + sback : -1, zmin, act);
        append_finish<1>(bins, &t1, &e);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// k_raster

template <int NT>
struct RasterLds {
  unsigned long long key[NT];  // packed (depth bits << 32 | face id)
  float ray[3][NT];            // ray_w of each tile pixel
  float fv[13][NT];            // staged faces: 3 projected verts, area, face normal
  int32_t fid[NT];
  uint16_t box[NT];            // lx0 | ly0 << 5 | (nx - 1) << 10 (tile-local pixel bbox)
  PairLds<NT> pairs;
  uint32_t flag[NT / 32];      // pixel saw a depth outside [FLT_MIN, inf] (bit per pixel)
  uint32_t wmax[NT / 64];       // per-wave max of the pixels' depth bits
  int32_t any_flag;
  int32_t item;
  int4 runseg[4];              // counters of the persistent block's current run
};

// Exact sequential z-buffer for one pixel (slow path): the result of the
// reference's update rule `if (d < FLT_MIN || z < d)` (rasterizer.cc:228-237),
// applied in increasing face id over the faces of the tile's bin that cover the
// pixel, starting from d = 0. Used only for pixels where some covering face
// produced a depth below FLT_MIN or NaN, where the packed atomicMin order is
// not the sequential order.
//
// Without NaN depths the rule has a closed form, computed in two passes over
// the bin: a covering face with depth below FLT_MIN is always taken, so the
// last such face E (largest id) resets the pixel, the next face is taken
// unconditionally, and from there the strict-less rule keeps the first
// smallest depth. The winner is therefore the smallest (depth, id) among the
// covering faces after E with depth >= FLT_MIN, or E itself when there is none.
// A NaN depth is taken only right after a reset and then blocks every later
// face; when a covering face has one, the rule is simulated in id order
// instead (one pass over the bin per covering face).
UGU_DEV void sequential_pixel(const DevView& v, const DevMesh& mesh,
                              const int2* bin, int nA, int cap, int n,
                              int gx, int gy, float r0, float r1, float r2,
                              int& out_fid) {
  const float x = static_cast<float>(gx), y = static_cast<float>(gy);
  // face of bin entry i and its depth at the pixel; false when it does not
  // cover the pixel
  auto covers = [&](int i, int& f, float& z) {
    f = bin_entry(bin, nA, cap, i).x;
    float P[9], N[3];
    load_face_rec(mesh.soup, f, P, N);
    const float4 a = project_point(v, P[0], P[1], P[2]);
    const float4 b = project_point(v, P[3], P[4], P[5]);
    const float4 c = project_point(v, P[6], P[7], P[8]);
    int x0, x1, y0, y1;
    float area;
    if (!face_setup(a, b, c, v.W, v.H, x0, x1, y0, y1, area)) return false;
    if (gx < x0 || gx > x1 || gy < y0 || gy > y1) return false;
    const bool bf = mesh.fnormals != nullptr && sum3(N[0] * r0, N[1] * r1, N[2] * r2) > 0.0f;
    float w0, w1, w2;
    return cover_test(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, area, bf, x, y, z, w0, w1,
                      w2);
  };
  // pass 1: the last reset face and whether any depth is NaN
  int emax = -1;
  bool any_nan = false;
  for (int i = 0; i < n; i++) {
    int f;
    float z;
    if (!covers(i, f, z)) continue;
    if (z != z) any_nan = true;
    else if (z < FLT_MIN) emax = max(emax, f);
  }
  if (!any_nan) {
    // pass 2: first smallest depth after the reset
    unsigned long long best = ~0ull;
    for (int i = 0; i < n; i++) {
      int f;
      float z;
      if (!covers(i, f, z) || f <= emax || !(z >= FLT_MIN)) continue;
      const unsigned long long key =
          (static_cast<unsigned long long>(__float_as_uint(z)) << 32) | static_cast<unsigned int>(f);
      best = key < best ? key : best;
    }
    out_fid = best != ~0ull ? static_cast<int>(best & 0xffffffffull) : emax;
    return;
  }
  // some depth is NaN: the rule in id order
  int cur = -1;
  float d = 0.0f;
  int dfid = -1;
  for (;;) {
    int best = INT_MAX;
    float bestz = 0.0f;
    for (int i = 0; i < n; i++) {
      int f;
      float z;
      if (covers(i, f, z) && f > cur && f < best) {
        best = f;
        bestz = z;
      }
    }
    if (best == INT_MAX) break;
    if (d < FLT_MIN || bestz < d) {
      d = bestz;
      dfid = best;
    }
    cur = best;
  }
  out_fid = dfid;
}


// Differentiable image model in float64 for one covered pixel: colour term times
// texture term (visibility comes from the float32 rasterizer; in double, so that
// the image matches the exact model, not the float32 rounding of thin triangles).
// With x, y the corners' camera positions sheared so that the pixel's ray is their
// z axis (x = fx Qx - (px - cx) Qz, y likewise), the perspective-correct weight of
// a corner is proportional to the cross product of the other two.
// The arrays are gathered by index: on a mesh of a face per pixel they are 40
// bytes a face, the face and shading records 112, and the gathers' L2 misses bound
// the pass (64 views of 1.3 M faces: 1011 against 1038 us). The model without the
// derivatives and without the corners' screen positions needs 40 float64
// operations instead of 130 and no spilled registers: 1003 -> 895 us. (In a kernel
// of its own after k_raster: 624 + 639 us.)
UGU_DEV void diff_image(const DevView& v, const DevMesh& m, int fid, int px, int py, float img[3]) {
#pragma clang fp contract(fast)
  int32_t vid[3], uid[3] = {0, 0, 0};
  for (int j = 0; j < 3; j++) vid[j] = m.faces[int64_t(fid) * 3 + j];
  if (m.ftex)
    for (int j = 0; j < 3; j++) uid[j] = m.uvidx[int64_t(fid) * 3 + j];
  const double u = px - static_cast<double>(v.cx), w = py - static_cast<double>(v.cy);
  double ax[4], ay[4];
  for (int k = 0; k < 4; k++) {
    const double c0 = k < 3 ? v.w2c_R[k] : v.trel[0], c1 = k < 3 ? v.w2c_R[3 + k] : v.trel[1],
                 c2 = k < 3 ? v.w2c_R[6 + k] : v.trel[2];
    ax[k] = v.fx * c0 - u * c2;
    ay[k] = v.fy * c1 - w * c2;
  }
  double X[3], Y[3];
  for (int j = 0; j < 3; j++) {
    const float* P = m.verts + int64_t(vid[j]) * 3;
    const double p0 = P[0] - v.org[0], p1 = P[1] - v.org[1], p2 = P[2] - v.org[2];
    X[j] = ax[0] * p0 + ax[1] * p1 + ax[2] * p2 + ax[3];
    Y[j] = ay[0] * p0 + ay[1] * p1 + ay[2] * p2 + ay[3];
  }
  const double q0 = X[2] * Y[1] - X[1] * Y[2];
  const double q1 = X[0] * Y[2] - X[2] * Y[0];
  const double q2 = X[1] * Y[0] - X[0] * Y[1];
  const double is = recip(q0 + q1 + q2);
  const double b1 = q1 * is, b2 = q2 * is, b0 = 1.0 - b1 - b2;
  double col[3] = {1.0, 1.0, 1.0};
  if (m.vcolors) {
    const float* ca = m.vcolors + int64_t(vid[0]) * 3;
    const float* cb = m.vcolors + int64_t(vid[1]) * 3;
    const float* cc = m.vcolors + int64_t(vid[2]) * 3;
    for (int k = 0; k < 3; k++) col[k] = b0 * ca[k] + b1 * cb[k] + b2 * cc[k];
  }
  if (m.ftex) {
    const float* ua = m.uv + int64_t(uid[0]) * 2;
    const float* ub = m.uv + int64_t(uid[1]) * 2;
    const float* uc = m.uv + int64_t(uid[2]) * 2;
    const double iu = b0 * ua[0] + b1 * ub[0] + b2 * uc[0];
    const double iv = b0 * ua[1] + b1 * ub[1] + b2 * uc[1];
    const int tw = m.ftex_w, th = m.ftex_h;
    const double fxp = iu * (tw - 1), fyp = (1.0 - iv) * (th - 1);
    const double flx = floor(fxp), fly = floor(fyp);
    const double lu = fxp - flx, lv = fyp - fly;
    const int tx0 = clamp_cell(flx, tw - 1), tx1 = clamp_cell(flx + 1.0, tw - 1);
    const int ty0 = clamp_cell(fly, th - 1), ty1 = clamp_cell(fly + 1.0, th - 1);
    const float* p00 = m.ftex + (int64_t(ty0) * tw + tx0) * 3;
    const float* p01 = m.ftex + (int64_t(ty0) * tw + tx1) * 3;
    const float* p10 = m.ftex + (int64_t(ty1) * tw + tx0) * 3;
    const float* p11 = m.ftex + (int64_t(ty1) * tw + tx1) * 3;
    for (int k = 0; k < 3; k++) {
      const double r0 = p00[k] + lu * (static_cast<double>(p01[k]) - p00[k]);
      const double r1 = p10[k] + lu * (static_cast<double>(p11[k]) - p10[k]);
      col[k] *= r0 + lv * (r1 - r0);
    }
  }
  for (int k = 0; k < 3; k++) img[k] = static_cast<float>(col[k]);
}

// G-buffer planes of one pixel (see UguGBuffer in ugu_hip.h). u, v: the
// winner's perspective-correct weights of its second and third vertex; P: its
// world vertex positions (null when no position plane is written); uvm: the
// mesh when the uv plane is written and the mesh has uvs; n: the shading normal.
template <bool STREAM>
UGU_DEV void write_gbuffer(const DevView& v, int64_t pidx, bool covered, float u, float vv,
                           bool has_p, const float* P, const DevMesh* uvm, float n0, float n1,
                           float n2, int fid = 0) {
  float b[3] = {0.0f, 0.0f, 0.0f}, t[3] = {0.0f, 0.0f, 0.0f};
  float pw[3] = {0.0f, 0.0f, 0.0f}, pc[3] = {0.0f, 0.0f, 0.0f};
  if (covered) {
    const float w = 1.0f - u - vv;
    b[0] = u;
    b[1] = vv;
    b[2] = 1.0f - u - vv;
    if (uvm) {
      const int32_t* ui = uvm->uvidx + int64_t(fid) * 3;
      const float* a = uvm->uv + int64_t(ui[0]) * 2;
      const float* bb = uvm->uv + int64_t(ui[1]) * 2;
      const float* c = uvm->uv + int64_t(ui[2]) * 2;
      t[0] = w * a[0] + u * bb[0] + vv * c[0];
      t[1] = w * a[1] + u * bb[1] + vv * c[1];
      t[2] = 1.0f - t[0] - t[1];
    }
    if (has_p) {
      for (int k = 0; k < 3; k++) pw[k] = w * P[k] + u * P[3 + k] + vv * P[6 + k];
      for (int r = 0; r < 3; r++)
        pc[r] = v.w2c_t[r] + sum3(v.w2c_R[r * 3 + 0] * pw[0], v.w2c_R[r * 3 + 1] * pw[1],
                                  v.w2c_R[r * 3 + 2] * pw[2]);
    }
  } else {
    n0 = n1 = n2 = 0.0f;
  }
  if (v.bary) put3<STREAM>(v.bary, pidx, b[0], b[1], b[2]);
  if (v.uvo) put3<STREAM>(v.uvo, pidx, t[0], t[1], t[2]);
  if (v.pos_wld) put3<STREAM>(v.pos_wld, pidx, pw[0], pw[1], pw[2]);
  if (v.pos_cam) put3<STREAM>(v.pos_cam, pidx, pc[0], pc[1], pc[2]);
  if (v.nrm_wld) put3<STREAM>(v.nrm_wld, pidx, n0, n1, n2);
  if (v.geo_id) put<STREAM>(v.geo_id, pidx, covered ? 0 : -1);
}

// One screen tile; `seg` is the tile's counter record (front count, back
// count, back-segment minimum skip depth, view index).
template <int TW, int TH, bool DIFF>
UGU_DEV void raster_tile(RasterLds<TW * TH>& s, int gtile, const int4 seg, const DevView* views,
                         const DevMesh& mesh,
                         const DevBins& bins, const DevOptions& opt) {
  constexpr int NT = TW * TH;
  // output planes streamed past L2 when the tile's rows are long enough
  constexpr bool S = TW >= 16;
  const int t = threadIdx.x;

  const int count = seg.x + seg.y;
  const DevView& v = views[seg.w];
  const int lt = gtile - v.tile_base;
  const int tyi = lt / v.tiles_x;
  const int txi = lt - tyi * v.tiles_x;
  const int px0 = txi * TW, py0 = tyi * TH;

  // this thread's pixel
  const int lx = t % TW, ly = t / TW;
  const int gx = px0 + lx, gy = py0 + ly;
  if (count == 0) {
    // no face touches the tile: every pixel keeps the initial values of
    // ValidateAndInitBeforeRender (util_private.cc:68-87)
    if (gx < v.W && gy < v.H) {
      const int64_t pidx = int64_t(gy) * v.W + gx;
      if (DIFF) {
        put3<S>(v.image, pidx, 0.0f, 0.0f, 0.0f);
        put<S>(v.face_id, pidx, -1);
        return;
      }
      if (v.color) put3<S>(v.color, pidx, uint8_t(0), uint8_t(0), uint8_t(0));
      if (v.depth) put<S>(v.depth, pidx, 0.0f);
      if (v.normal) put3<S>(v.normal, pidx, 0.0f, 0.0f, 0.0f);
      if (v.mask) put<S>(v.mask, pidx, uint8_t(0));
      write_gbuffer<S>(v, pidx, false, 0.0f, 0.0f, false, nullptr, nullptr, 0.0f, 0.0f, 0.0f);
      if (v.face_id) put<S>(v.face_id, pidx, -1);
    }
    return;
  }
  // front segment first, then the back segment (both clipped to the bin)
  const int nA = seg.x < bins.cap ? seg.x : bins.cap;
  const int nB = seg.y < bins.cap - nA ? seg.y : bins.cap - nA;
  const int n = nA + nB;
  const int2* bin = bins.bins + int64_t(gtile) * bins.cap;
  // the first chunk's entries are loaded while the rays are computed; every
  // chunk then loads the next chunk's entries before its own pairs
  const int chunks_a = (nA + NT - 1) / NT, chunks = chunks_a + (nB + NT - 1) / NT;
  int2 e_next = make_int2(0, 0);
  if (t < (chunks_a > 0 ? nA : n)) e_next = bin_entry(bin, nA, bins.cap, t);

  // the rays stay in LDS: 72 registers leave no room for them in the pair loop
  {
    float r0, r1, r2;
    ray_w_at(v, static_cast<float>(gx), static_cast<float>(gy), r0, r1, r2);
    s.ray[0][t] = r0;
    s.ray[1][t] = r1;
    s.ray[2][t] = r2;
  }
  s.key[t] = ~0ull;
  if (t < NT / 32) s.flag[t] = 0u;
  if (t == 0) s.any_flag = 0;
  // When face ids fit 24 bits the depth key also carries the LDS slot of the
  // face (below the id, so ties still go to the lowest id). After every chunk
  // each thread copies the staged record of its pixel's current winner into
  // registers when the winner changed, so the resolve needs no second gather
  // and projection of the winning face.
  static_assert(NT <= 256, "slot keys hold 8-bit LDS slots");
  const bool slot_key = mesh.F <= (1 << 24);
  unsigned long long seen = ~0ull;  // key whose coverage the registers hold
  float wz = 0.0f, ww0 = 0.0f, ww1 = 0.0f, ww2 = 0.0f;
  bool wbf = false;
  // overflowing tiles report their true occupancy; the host re-renders with
  // bins that large (one same-address atomic per overflowing tile only)
  if (t == 0 && count > bins.cap) {
    atomicMax(&bins.status[0], count);
    *bins.host_flag = 1;
  }
  __syncthreads();

  // Largest depth any in-view pixel of the tile holds after the previous
  // chunks (NaN while some pixel has none). Keys only decrease, so a face
  // whose skip depth exceeds it is dropped before it is fetched. The back
  // segment starts a new chunk so that all of its faces are tested against
  // the depths the front faces left.
  float dmax = __uint_as_float(0xffffffffu);
  for (int ch = 0; ch < chunks; ch++) {
    // the whole back segment is skipped when even its smallest skip depth
    // exceeds the tile's depth bound
    if (ch == chunks_a && skip_face(__uint_as_float(static_cast<uint32_t>(seg.z)), dmax)) break;
    const int base = ch < chunks_a ? ch * NT : nA + (ch - chunks_a) * NT;
    const int end = ch < chunks_a ? nA : n;
    const bool more = ch + 1 < chunks;
    const int i = base + t;
    const int2 e = e_next;
    if (more) {
      const int nbase = ch + 1 < chunks_a ? (ch + 1) * NT : nA + (ch + 1 - chunks_a) * NT;
      const int nend = ch + 1 < chunks_a ? nA : n;
      e_next = nbase + t < nend ? bin_entry(bin, nA, bins.cap, nbase + t) : make_int2(0, 0);
    }
    // stage one chunk of faces
    int c = 0;
    if (i < end && !skip_face(__int_as_float(e.y), dmax)) {
      const int f = e.x;
      float P[9], N[3];
      load_face_rec(mesh.soup, f, P, N);
      const float4 a = project_point(v, P[0], P[1], P[2]);
      const float4 b = project_point(v, P[3], P[4], P[5]);
      const float4 cc = project_point(v, P[6], P[7], P[8]);
      int x0, x1, y0, y1;
      float area;
      if (face_setup(a, b, cc, v.W, v.H, x0, x1, y0, y1, area)) {
        const int lx0 = max(x0, px0) - px0, lx1 = min(x1, px0 + TW - 1) - px0;
        const int ly0 = max(y0, py0) - py0, ly1 = min(y1, py0 + TH - 1) - py0;
        if (lx0 <= lx1 && ly0 <= ly1) {
          const int nx = lx1 - lx0 + 1;
          c = nx * (ly1 - ly0 + 1);
          s.box[t] = static_cast<uint16_t>(lx0 | (ly0 << 5) | ((nx - 1) << 10));
        }
      }
      s.fv[0][t] = a.x; s.fv[1][t] = a.y; s.fv[2][t] = a.z;
      s.fv[3][t] = b.x; s.fv[4][t] = b.y; s.fv[5][t] = b.z;
      s.fv[6][t] = cc.x; s.fv[7][t] = cc.y; s.fv[8][t] = cc.z;
      s.fv[9][t] = area;
      s.fv[10][t] = N[0]; s.fv[11][t] = N[1]; s.fv[12][t] = N[2];
      s.fid[t] = f;
    }
    publish_pairs(s.pairs, ch & 1, c);
    __syncthreads();
    const bool has_fn = mesh.fnormals != nullptr;
    // One (face slot, tile pixel) pair: coverage, depth and the packed LDS
    // atomicMin.
    auto test_pair = [&](int j, int pix) {
      const int pxl = static_cast<int>(static_cast<unsigned>(pix) % TW);
      const int pyl = static_cast<int>(static_cast<unsigned>(pix) / TW);
      const float rx = s.ray[0][pix], ry = s.ray[1][pix], rz = s.ray[2][pix];
      const bool bf = has_fn && sum3(s.fv[10][j] * rx, s.fv[11][j] * ry, s.fv[12][j] * rz) > 0.0f;
      float z, w0, w1, w2;
      if (cover_test(s.fv[0][j], s.fv[1][j], s.fv[2][j], s.fv[3][j], s.fv[4][j],
                     s.fv[5][j], s.fv[6][j], s.fv[7][j], s.fv[8][j], s.fv[9][j],
                     bf, static_cast<float>(px0 + pxl), static_cast<float>(py0 + pyl),
                     z, w0, w1, w2)) {
        if (z >= FLT_MIN) {
          const unsigned int lowbits =
              slot_key ? (static_cast<unsigned int>(s.fid[j]) << 8) | static_cast<unsigned int>(j)
                       : static_cast<unsigned int>(s.fid[j]);
          const unsigned long long key =
              (static_cast<unsigned long long>(__float_as_uint(z)) << 32) | lowbits;
          atomicMin(&s.key[pix], key);
        } else {
          atomicOr(&s.flag[pix >> 5], 1u << (pix & 31));
          s.any_flag = 1;
        }
      }
    };
    // Most pairs of a box are not covered: a pair first needs edge functions of
    // one sign (cover_test's, same bits; a NaN only keeps it), and the pairs
    // that pass are tested 64 at a time.
    auto one_sign = [&](int j, int r, int& pix) {
      const int bx = s.box[j];
      const int nx = (bx >> 10) + 1;
      const int qy = pair_row(r, nx);
      const int pxl = (bx & 31) + (r - qy * nx), pyl = ((bx >> 5) & 31) + qy;
      pix = pyl * TW + pxl;
      const float x = static_cast<float>(px0 + pxl), y = static_cast<float>(py0 + pyl);
      const float ax = s.fv[0][j], ay = s.fv[1][j], bx_ = s.fv[3][j], by = s.fv[4][j],
                  cx = s.fv[6][j], cy = s.fv[7][j];
      const float w0 = edge_fn(bx_, by, cx, cy, x, y);
      const float w1 = edge_fn(cx, cy, ax, ay, x, y);
      const float w2 = edge_fn(ax, ay, bx_, by, x, y);
      return fminf(fminf(w0, w1), w2) >= 0.0f || fmaxf(fmaxf(w0, w1), w2) <= 0.0f;
    };
    // a chunk without any pair (every face skipped or off the tile) ends here
    if (walk_pairs(s.pairs, ch & 1, one_sign, test_pair) == 0) continue;
    __syncthreads();
    const unsigned long long k = s.key[t];
    if (more) {
      // depth bits of this pixel: all ones when it has no key yet, 0 outside
      // the image (no face reaches those pixels)
      uint32_t db = (gx < v.W && gy < v.H) ? static_cast<uint32_t>(k >> 32) : 0u;
      db = wave_max_u32(db);
      if ((t & 63) == 0) s.wmax[t >> 6] = db;
    }
    if (slot_key && k != seen) {
      // the pixel's winner changed: evaluate its coverage from the staged
      // record with the pair test's arithmetic (same bits), so the resolve
      // needs neither the record nor a second test
      const int sl = static_cast<int>(k & 0xffull);
      wbf = has_fn && sum3(s.fv[10][sl] * s.ray[0][t], s.fv[11][sl] * s.ray[1][t],
                           s.fv[12][sl] * s.ray[2][t]) > 0.0f;
      cover_test(s.fv[0][sl], s.fv[1][sl], s.fv[2][sl], s.fv[3][sl], s.fv[4][sl], s.fv[5][sl],
                 s.fv[6][sl], s.fv[7][sl], s.fv[8][sl], s.fv[9][sl], wbf,
                 static_cast<float>(gx), static_cast<float>(gy), wz, ww0, ww1, ww2);
      seen = k;
    }
    if (more) {
      // the next chunk's staging overwrites the records read above
      __syncthreads();
      uint32_t m = s.wmax[0];
      for (int w = 1; w < NT / 64; w++) m = max(m, s.wmax[w]);
      dmax = __uint_as_float(m);
    }
  }

  // ---- resolve (rasterizer.cc:243-301) for this thread's pixel; the
  // winner's depth, weights and back-face flag are in registers (slot keys)
  // or computed again below
  const float r0 = s.ray[0][t], r1 = s.ray[1][t], r2 = s.ray[2][t];
  int fid = -1;
  bool have = false;
  if (s.any_flag && ((s.flag[t >> 5] >> (t & 31)) & 1u)) {
    sequential_pixel(v, mesh, bin, nA, bins.cap, n, gx, gy, r0, r1, r2, fid);
  } else if (seen != ~0ull) {
    fid = static_cast<int>(static_cast<unsigned int>(seen & 0xffffffffull) >> 8);
    have = true;
  } else if (!slot_key) {
    const unsigned long long key = s.key[t];
    if (key != ~0ull) fid = static_cast<int>(key & 0xffffffffull);
  }
  __syncthreads();  // LDS is reused by the next tile of a persistent block
  if (gx >= v.W || gy >= v.H) return;

  float z = 0.0f, w0 = 0.0f, w1 = 0.0f, w2 = 0.0f;
  bool bf = false;
  if (fid >= 0) {
    if (have) {
      z = wz;
      w0 = ww0;
      w1 = ww1;
      w2 = ww2;
      bf = wbf;
    } else {
      float P[9], N[3];
      load_face_rec(mesh.soup, fid, P, N);
      const float4 a = project_point(v, P[0], P[1], P[2]);
      const float4 b = project_point(v, P[3], P[4], P[5]);
      const float4 c = project_point(v, P[6], P[7], P[8]);
      const float area = edge_fn(a.x, a.y, b.x, b.y, c.x, c.y);
      bf = mesh.fnormals != nullptr && sum3(N[0] * r0, N[1] * r1, N[2] * r2) > 0.0f;
      cover_test(a.x, a.y, a.z, b.x, b.y, b.z, c.x, c.y, c.z, area, bf,
                 static_cast<float>(gx), static_cast<float>(gy), z, w0, w1, w2);
    }
    if (opt.culling && bf) {
      fid = -1;
      z = 0.0f;
    }
  }
  const int64_t pidx = int64_t(gy) * v.W + gx;

  if (DIFF) {
    // differentiable forward: image = colour term * texture term (float64)
    float img[3] = {0.0f, 0.0f, 0.0f};
    if (fid > 0) diff_image(v, mesh, fid, gx, gy, img);
    put3<S>(v.image, pidx, img[0], img[1], img[2]);
    put<S>(v.face_id, pidx, fid);
  } else {
    uint8_t col[3] = {0, 0, 0};
    float nrm[3] = {0.0f, 0.0f, 0.0f};
    uint8_t msk = 0;
    const bool gbuf = v.bary || v.uvo || v.pos_wld || v.pos_cam || v.nrm_wld || v.geo_id;
    if (fid > 0) msk = 255;
    if (fid > 0 && (v.color || v.normal || gbuf)) {
      float n0, n1, n2;
      FaceShade fs;
      face_shade(mesh, fid, opt.shading_normal != 0, v.color && opt.diffuse_color == 1, fs);
      if (opt.shading_normal == 0) {
        const float* fn = mesh.fnormals + int64_t(fid) * 3;
        n0 = fn[0]; n1 = fn[1]; n2 = fn[2];
      } else {
        const float* na = fs.na;
        const float* nb = fs.nb;
        const float* nc = fs.nc;
        n0 = w0 * na[0] + w1 * nb[0] + w2 * nc[0];
        n1 = w0 * na[1] + w1 * nb[1] + w2 * nc[1];
        n2 = w0 * na[2] + w1 * nb[2] + w2 * nc[2];
      }
      if (v.normal) {
        nrm[0] = sum3(v.w2c_R[0] * n0, v.w2c_R[1] * n1, v.w2c_R[2] * n2);
        nrm[1] = sum3(v.w2c_R[3] * n0, v.w2c_R[4] * n1, v.w2c_R[5] * n2);
        nrm[2] = sum3(v.w2c_R[6] * n0, v.w2c_R[7] * n1, v.w2c_R[8] * n2);
      }
      if (v.color) shade_u8(mesh, opt, fid, fs, w1, w2, r0, r1, r2, n0, n1, n2, col);
      if (gbuf) {
        // P is passed with a flag, not as a pointer that may be null: a select
        // between pointers would keep the array out of registers
        float P[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, N[3];
        const bool pos = v.pos_wld || v.pos_cam;
        if (pos) load_face_rec(mesh.soup, fid, P, N);
        write_gbuffer<S>(v, pidx, true, w1, w2, pos, P,
                         v.uvo && mesh.uv && mesh.uvidx ? &mesh : nullptr, n0, n1, n2, fid);
      }
    } else if (gbuf) {
      write_gbuffer<S>(v, pidx, false, 0.0f, 0.0f, false, nullptr, nullptr, 0.0f, 0.0f, 0.0f);
    }
    if (v.color) put3<S>(v.color, pidx, col[0], col[1], col[2]);
    if (v.depth) put<S>(v.depth, pidx, z);
    if (v.normal) put3<S>(v.normal, pidx, nrm[0], nrm[1], nrm[2]);
    if (v.mask) put<S>(v.mask, pidx, msk);
    if (v.face_id) put<S>(v.face_id, pidx, fid);
  }
  // The tile's counters, cleared for the next pass (an empty tile's are clear).
  // Last: a wavefront's later loads wait for an earlier store, and here none
  // follow (after the first barrier the store cost the 64-view step 50 us).
  if (t == 0) reinterpret_cast<int4*>(bins.counts)[gtile] = make_int4(0, 0, 0x7f800000, seg.w);
}

template <int TW, int TH, bool DIFF>
// A tile is a chain of dependent steps (counters, entries, face records, pairs,
// the winners' shading inputs): a pass of one view ends with its slowest tile, a
// pass of many is bound by how many tiles are in flight. So 7 waves per SIMD for
// rendering (72 VGPRs; 7 blocks of 22.7 KB fill the 160 KB of LDS); the
// differentiable forward needs 91 VGPRs and takes 5 (6 would spill: 896 against
// 911 us for the case below).
// Slowest tile of 1.3 M faces at 1080p: 130,000 cycles with its faces' pairs
// written one by one by the faces' threads (93,000 of them in the pairs, silhouette
// slivers), 65 -> 46 us for the kernel with walk_pairs; 640x480, 32 k faces:
// 35 -> 22 us. 64 mixed views: 825 -> 815 us; differentiable forward of them
// 1003 -> 895 us.
__global__ __launch_bounds__(TW * TH, DIFF ? 5 : 7) void k_raster(
    const DevView* __restrict__ views, DevMesh mesh,
    DevBins bins, DevOptions opt,
    int persistent) {
  __shared__ RasterLds<TW * TH> s;
  if (!persistent) {
    const int gtile = xcd_remap(blockIdx.x, gridDim.x);
    raster_tile<TW, TH, DIFF>(s, gtile, reinterpret_cast<const int4*>(bins.counts)[gtile], views,
                              mesh, bins, opt);
    return;
  }
  // persistent: pull runs of kQueueRun consecutive (view, tile) items until
  // every queue is drained. Run r belongs to queue r % kQueues; a block starts
  // at queue blockIdx.x % kQueues and, once that one is drained, takes the
  // next queue's runs. Each head only grows and every run below n_runs is
  // handed out once, so a block that finds all kQueues heads past their
  // runs (one atomic each, at most kQueues in a row) leaves with every run
  // claimed. The next run is claimed when the last tile of the current one
  // starts. The barrier before reading s.item publishes thread 0's write (an
  // empty tile returns from raster_tile without a barrier); the one after
  // keeps thread 0 from overwriting it before every thread has read it.
  // `item` is the same in every thread, so every thread leaves the loop
  // together. The counter records of a run's tiles are read together into
  // LDS, one round trip per run (most tiles of a batch are empty and need
  // nothing else).
  constexpr int kQueueRun = 2;
  static_assert(kQueueRun <= 4, "RasterLds::runseg holds one run");
  const int n_runs = (bins.total_tiles + kQueueRun - 1) / kQueueRun;
  int queue = static_cast<int>(blockIdx.x % kQueues);  // used by thread 0
  auto claim = [&]() {
    for (int k = 0; k < kQueues; k++) {
      const int r = atomicAdd(&bins.status[kQueueStride * (queue + 1)], 1);
      if (r < (n_runs - queue + kQueues - 1) / kQueues) return (queue + kQueues * r) * kQueueRun;
      queue = (queue + 1) % kQueues;
    }
    return bins.total_tiles;
  };
  if (threadIdx.x == 0) s.item = claim();
  __syncthreads();
  int item = s.item;
  __syncthreads();
  while (item < bins.total_tiles) {
    const int end = min(item + kQueueRun, bins.total_tiles);
    if (threadIdx.x < end - item)
      s.runseg[threadIdx.x] = reinterpret_cast<const int4*>(bins.counts)[item + threadIdx.x];
    __syncthreads();
    for (int it = item; it < end; it++) {
      if (it == end - 1 && threadIdx.x == 0) s.item = claim();
      raster_tile<TW, TH, DIFF>(s, it, s.runseg[it - item], views, mesh, bins, opt);
    }
    __syncthreads();
    item = s.item;
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// RenderW depth conversion: uint16(1.0 * (double)d), truncating as x86 does.
__global__ void k_depth_to_u16(const float* __restrict__ d, int64_t n,
                               uint16_t* __restrict__ out) {
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = 1.0 * static_cast<double>(d[i]);
  int32_t iv = (s >= -2147483648.0 && s < 2147483648.0) ? static_cast<int32_t>(s) : INT32_MIN;
  out[i] = static_cast<uint16_t>(static_cast<uint32_t>(iv) & 0xffffu);
}

// ---------------------------------------------------------------------------
// host-side launchers (called from ugu_hip.cpp)

// hv: the host descriptors of n_views <= kInlineViews views, written to `views`;
// null: `views` holds them already. counts / status: null when the pass has none.
int launch_begin(hipStream_t st, const DevView* hv, int n_views, DevView* views, int32_t* counts,
                 int32_t n_tiles, int32_t* status) {
  const dim3 grid((n_tiles > 256 ? n_tiles + 255 : 256) / 256);
  if (hv && n_views == 1) {
    InlineViews<1> a;
    a.v[0] = hv[0];
    hipLaunchKernelGGL(k_begin<1>, grid, dim3(256), 0, st, a, nullptr, views, n_views, counts, n_tiles,
                       status);
  } else if (hv) {
    InlineViews<kInlineViews> a;
    for (int k = 0; k < n_views; k++) a.v[k] = hv[k];
    hipLaunchKernelGGL(k_begin<kInlineViews>, grid, dim3(256), 0, st, a, nullptr, views, n_views,
                       counts, n_tiles, status);
  } else {
    hipLaunchKernelGGL(k_begin<0>, grid, dim3(256), 0, st, InlineViews<1>{}, views, nullptr, n_views,
                       counts, n_tiles, status);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_shade_rec(hipStream_t st, const DevMesh& m, float4* out) {
  if (m.F <= 0) return 0;
  hipLaunchKernelGGL(k_shade_rec, dim3((m.F + 255) / 256), dim3(256), 0, st, m, out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_face_soup(hipStream_t st, const float* verts, const int32_t* faces,
                     const float* fnormals, int32_t F, int compute_normals, float4* soup,
                     float* fn_out) {
  if (F <= 0) return 0;
  hipLaunchKernelGGL(k_face_soup, dim3((F + 255) / 256), dim3(256), 0, st, verts, faces,
                     fnormals, F, compute_normals, soup, fn_out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// one: the host descriptor of a pass of one view whose counters are clear (no
// launch_begin), written to `views`; otherwise null
int launch_setup_bin(hipStream_t st, int tw, int th, const DevView* one, DevView* views,
                     int n_views, const DevMesh& mesh,
                     const DevBins& bins) {
  if (mesh.F <= 0) return 0;
  dim3 grid((mesh.F + 255) / 256, (n_views + kSetupViews - 1) / kSetupViews), block(256);
  InlineViews<1> a{};
  if (one) a.v[0] = *one;
#define UGU_SETUP_CASE(TWV, THV)                                                          \
  if (tw == TWV && th == THV) {                                                           \
    if (one)                                                                              \
      hipLaunchKernelGGL((k_setup_bin<TWV, THV, true>), grid, block, 0, st, a, nullptr,   \
                         views, 1, mesh, bins);                                           \
    else                                                                                  \
      hipLaunchKernelGGL((k_setup_bin<TWV, THV, false>), grid, block, 0, st, a, views,    \
                         nullptr, n_views, mesh, bins);                                   \
    return hipGetLastError() == hipSuccess ? 0 : -1;                                      \
  }
  UGU_SETUP_CASE(8, 8)
  UGU_SETUP_CASE(16, 16)
  UGU_SETUP_CASE(32, 8)
#undef UGU_SETUP_CASE
  return -2;
}

template <bool DIFF>
static int launch_raster_t(hipStream_t st, int tw, int th, const DevView* views,
                           const DevMesh& mesh, const DevBins& bins, const DevOptions& opt,
                           int persistent_blocks) {
  const int grid = persistent_blocks > 0 ? persistent_blocks : bins.total_tiles;
#define UGU_RASTER_CASE(TWV, THV)                                                              \
  if (tw == TWV && th == THV) {                                                                \
    hipLaunchKernelGGL((k_raster<TWV, THV, DIFF>), dim3(grid), dim3(TWV * THV), 0, st, views,  \
                       mesh, bins, opt, persistent_blocks > 0 ? 1 : 0);                        \
    return hipGetLastError() == hipSuccess ? 0 : -1;                                           \
  }
  UGU_RASTER_CASE(8, 8)
  UGU_RASTER_CASE(16, 16)
  UGU_RASTER_CASE(32, 8)
#undef UGU_RASTER_CASE
  return -2;
}

int launch_raster(hipStream_t st, int tw, int th, int mode, const DevView* views,
                  const DevMesh& mesh, const DevBins& bins, const DevOptions& opt,
                  int persistent_blocks) {
  if (bins.total_tiles <= 0) return 0;
  return mode == 0
             ? launch_raster_t<false>(st, tw, th, views, mesh, bins, opt, persistent_blocks)
             : launch_raster_t<true>(st, tw, th, views, mesh, bins, opt, persistent_blocks);
}

template <bool DIFF>
static int raster_occupancy(int tw, int th) {
  int nb = 0;
  hipError_t e = hipErrorInvalidValue;
#define UGU_OCC_CASE(TWV, THV)                                                               \
  if (tw == TWV && th == THV)                                                                \
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_raster<TWV, THV, DIFF>, TWV * THV, 0);
  UGU_OCC_CASE(8, 8)
  UGU_OCC_CASE(16, 16)
  UGU_OCC_CASE(32, 8)
#undef UGU_OCC_CASE
  return e == hipSuccess ? nb : 0;
}

int raster_blocks_per_cu(int tw, int th, int mode) {
  return mode == 0 ? raster_occupancy<false>(tw, th) : raster_occupancy<true>(tw, th);
}

int launch_depth_to_u16(hipStream_t st, const float* d, int64_t n, uint16_t* out) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(k_depth_to_u16, dim3((n + 255) / 256), dim3(256), 0, st, d, n, out);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugu_hip
