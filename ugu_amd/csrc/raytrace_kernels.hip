// HIP kernel of the gfx950 raytracer: Raytracer::Impl::Render
// (src/renderer/cpu/raytracer.cc:117-225) for a batch of views.
//
// Two ways to the same closest hit, both by the reference's float64
// Moller-Trumbore routine (src/util/geom_util.cc:60-115, epsilon double(1e-8f) of
// bvh_naive.h:121, standard barycentric conversion):
//   k_rt_setup, k_rt_tiles  bins of faces per 16x16 pixel tile, every ray tested
//                           against its tile's faces (meshes of few layers);
//   k_raytrace              one wave per 8x8 pixel tile walks the BVH (built on
//                           the host, nodes hold both children's boxes) as one
//                           packet of 64 rays, nearer child first, and every
//                           lane tests the triangles of every leaf reached.
// The closest hit is the smallest float t; equal t resolve to the lowest face
// id. The box test is float32 with widened boxes and a relative slack on the
// ray interval, so it only prunes boxes that cannot hold a hit the float64 test
// would accept; the bins' bounds are those of project_ray. Then the pixel is
// culled or shaded as in raytracer.cc:160-218.

#include "binning.h"
#include "device_common.h"
#include "rt_math.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace ugu_hip {

// Writes pixel (x, y): face bf hit at distance bt with the raytracer's weights
// (bu, bv), or no hit (bf < 0); culling, depth, normal and colour of
// raytracer.cc:160-218.
template <bool STREAM>
UGU_DEV void write_hit(const DevView& v, const DevMesh& m, const DevOptions& o, int x, int y, int bf,
                       float bt, float bu, float bv, float r0, float r1, float r2) {
  const int64_t pi = int64_t(y) * v.W + x;
  bool hit = bf >= 0;
  // back-face culling: face normal . ray_w > 0 -> background (raytracer.cc:166-172)
  if (hit && o.culling && backface_of(m.fnormals, bf, r0, r1, r2)) hit = false;
  if (!hit) {
    if (v.color) put3<STREAM>(v.color, pi, uint8_t(0), uint8_t(0), uint8_t(0));
    if (v.depth) put<STREAM>(v.depth, pi, 0.0f);
    if (v.normal) put3<STREAM>(v.normal, pi, 0.0f, 0.0f, 0.0f);
    if (v.mask) put<STREAM>(v.mask, pi, uint8_t(0));
    if (v.face_id) put<STREAM>(v.face_id, pi, -1);
    return;
  }
  // hit_pos_c = w2c_R * (org + ray * t) + w2c_t; depth = z * depth_scale
  const float h0 = v.c2w_t[0] + r0 * bt, h1 = v.c2w_t[1] + r1 * bt, h2 = v.c2w_t[2] + r2 * bt;
  const float zc = sum3(v.w2c_R[6] * h0, v.w2c_R[7] * h1, v.w2c_R[8] * h2) + v.w2c_t[2];
  float n0, n1, n2;
  FaceShade fs;
  face_shade(m, bf, o.shading_normal != 0, v.color && o.diffuse_color == 1, fs);
  if (o.shading_normal == 0) {
    const float* fn = m.fnormals + int64_t(bf) * 3;
    n0 = fn[0];
    n1 = fn[1];
    n2 = fn[2];
  } else {
    // (1 - u - v) n[i0] + u n[i1] + v n[i2] with the raytracer's (u, v)
    const float* na = fs.na;
    const float* nb = fs.nb;
    const float* nc = fs.nc;
    const float w = 1.0f - bu - bv;
    n0 = w * na[0] + bu * nb[0] + bv * nc[0];
    n1 = w * na[1] + bu * nb[1] + bv * nc[1];
    n2 = w * na[2] + bu * nb[2] + bv * nc[2];
  }
  if (v.color) {
    uint8_t c[3];
    shade_u8(m, o, bf, fs, bu, bv, r0, r1, r2, n0, n1, n2, c);
    put3<STREAM>(v.color, pi, c[0], c[1], c[2]);
  }
  if (v.depth) put<STREAM>(v.depth, pi, zc * o.depth_scale);
  if (v.normal)
    put3<STREAM>(v.normal, pi, sum3(v.w2c_R[0] * n0, v.w2c_R[1] * n1, v.w2c_R[2] * n2),
                 sum3(v.w2c_R[3] * n0, v.w2c_R[4] * n1, v.w2c_R[5] * n2),
                 sum3(v.w2c_R[6] * n0, v.w2c_R[7] * n1, v.w2c_R[8] * n2));
  if (v.mask) put<STREAM>(v.mask, pi, uint8_t(255));
  if (v.face_id) put<STREAM>(v.face_id, pi, bf);
}

// Four waves per workgroup, each on its own tile (no cross-wave sharing).
constexpr int kRtWaves = 4;

// One wave traces the 64 rays of an 8x8 pixel tile through the hierarchy
// together: the node and leaf indices are wave-uniform (fetched with scalar
// loads), every lane tests its own ray against the node's two child boxes,
// and a child is entered when any lane's ray may reach it (nearer child first
// by a vote of the lanes). The stack of deferred children is one LDS word per
// level for the whole wave. Each lane keeps its own closest hit, and the
// closest hit does not depend on the visiting order, so the result is the
// per-ray one; the traversal only decides which tests are made.

__global__ __launch_bounds__(64 * kRtWaves) void k_raytrace(const DevView* __restrict__ views,
                                                            const BvhNode* __restrict__ nodes,
                                                            const int2* __restrict__ leaves,
                                                            const float4* __restrict__ tris,
                                                            int n_views, int total_tiles,
                                                            int chunk, DevMesh m,
                                                            DevOptions o) {
  __shared__ int32_t stacks[kRtWaves][kBvhStack];
  const int wave = threadIdx.x >> 6;
  int32_t* stack = stacks[wave];
  // Tiles of all views are numbered consecutively (views[i].tile_base).
  // Workgroups go round-robin over the 8 XCDs; each XCD here takes runs of
  // `chunk` consecutive workgroups (neighbouring tiles share its L2), and the
  // runs alternate over the XCDs. The grid is a multiple of 8 chunk
  // workgroups, which makes the mapping a permutation.
  const int i = blockIdx.x;
  const int k = i >> 3;
  const int lb = (((k / chunk) << 3) + (i & 7)) * chunk + (k % chunk);
  const int g = lb * kRtWaves + wave;
  if (g >= total_tiles) return;  // uniform over the wave
  int lo = 0, hi = n_views - 1;  // last view with tile_base <= g
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (views[mid].tile_base <= g) lo = mid; else hi = mid - 1;
  }
  const DevView& v = views[lo];
  const int tiles_x = (v.W + 7) >> 3;
  const int tile = g - v.tile_base;
  const int lane = threadIdx.x & 63;
  const int x = (tile % tiles_x) * 8 + (lane & 7);
  const int y = (tile / tiles_x) * 8 + (lane >> 3);
  const bool act = x < v.W && y < v.H;

  // ray_w / org_ray_w tables (camera.h:482-513)
  float r0, r1, r2;
  ray_w_at(v, static_cast<float>(act ? x : 0), static_cast<float>(act ? y : 0), r0, r1, r2);
  const float ox = v.c2w_t[0], oy = v.c2w_t[1], oz = v.c2w_t[2];
  const float ix = 1.0f / r0, iy = 1.0f / r1, iz = 1.0f / r2;
  const double dox = ox, doy = oy, doz = oz, ddx = r0, ddy = r1, ddz = r2;
  const float kInf = __builtin_huge_valf();

  float bt = kInf, bu = 0.0f, bv = 0.0f;
  float tmax = kInf;  // box_tmax(bt), updated with bt
  int bf = -1;
  int sp = 0;
  int ref = 0;  // the root is inner node 0
  // Inner references point to larger node indices and every node is entered
  // at most once, so the walk ends; the builder bounds the depth, and with it
  // the stack, by kBvhStack.
  for (;;) {
    if (ref >= 0) {
      const BvhNode nd = nodes[ref];
      const int ra = __float_as_int(nd.a_lo.w), rb = __float_as_int(nd.b_lo.w);
      // both tests on every lane (no branch between the node's loads), then
      // inactive lanes and the empty child are masked out
      const float ea = box_entry(nd.a_lo, nd.a_hi, ox, oy, oz, ix, iy, iz, tmax);
      const float eb = box_entry(nd.b_lo, nd.b_hi, ox, oy, oz, ix, iy, iz, tmax);
      const float ta = act ? ea : kInf;
      const float tb = (act && rb != kBvhEmpty) ? eb : kInf;
      const bool ha = __any(ta != kInf), hb = __any(tb != kInf);
      if (ha && hb) {
        const int va = __popcll(__ballot(ta < tb)), vb = __popcll(__ballot(tb < ta));
        const bool a_first = va >= vb;
        stack[sp] = a_first ? rb : ra;
        sp++;
        ref = a_first ? ra : rb;
        continue;
      }
      if (ha || hb) {
        ref = ha ? ra : rb;
        continue;
      }
    } else {
      const int2 lf = leaves[~ref];
      for (int k = 0; k < lf.y; k++) {
        const float4* tr = tris + int64_t(lf.x + k) * 3;
        const float4 p0 = tr[0], p1 = tr[1], p2 = tr[2];
        float t, u, w;
        if (act && mt_hit(dox, doy, doz, ddx, ddy, ddz, p0, p1, p2, t, u, w)) {
          const int f = __float_as_int(p0.w);
          if (t < bt || (t == bt && f < bf)) {
            bt = t;
            bu = u;
            bv = w;
            bf = f;
            tmax = box_tmax(bt);
          }
        }
      }
    }
    if (sp == 0) break;
    sp--;
    ref = __builtin_amdgcn_readfirstlane(stack[sp]);
  }
  if (!act) return;
  write_hit<false>(v, m, o, x, y, bf, bt, bu, bv, r0, r1, r2);
}

// ---------------------------------------------------------------------------
// Binned path. All rays of a view start at the camera, so the face a pixel's
// ray hits first can be found as a rasterizer finds it: every face is put into
// the bins of the screen tiles its hits can lie in, and a tile tests its rays
// against its bin's faces only. The hit test is the same float64 one
// (mt_hit), so the closest hit is the hierarchy walk's; the bins only decide
// which tests are made, and they are conservative (project_ray).

// Pixel position of a world point as the rays see it: the ray of pixel (x, y)
// is c2w_R times the normalized ((x - cx) / fx, (y - cy) / fy, 1), so a point P
// lies on it where q = inverse(c2w_R) (P - c2w_t) is a multiple of that
// vector. Returns (x, y, q.z, w): rays of pixels further than w from (x, y) in
// x or y miss the point. w bounds the float32 rounding of this projection and
// of the rays: with u = 2^-24, S = |P - o| in the 1-norm and K the condition
// number of c2w_R, rays and q carry less than 25 u K S of absolute error (one
// rounding of P - o, of the matrix entries and of each product and sum, the
// same for the ray, whose normalization scales it as a whole); rt_rel is
// 64 u K, and an error dq of q moves the pixel by at most
// |dq| / q.z (f + |x - cx| + |y - cy|). The last roundings of x and y are
// 2^-20 of the same sum and of cx, cy (rt_abs). Points closer to the camera's
// plane than S / 64, behind it or not finite get w = -1: no bound.
UGU_DEV float4 project_ray(const DevView& v, float px, float py, float pz) {
  const float dx = px - v.c2w_t[0], dy = py - v.c2w_t[1], dz = pz - v.c2w_t[2];
  const float qx = v.inv[0] * dx + v.inv[1] * dy + v.inv[2] * dz;
  const float qy = v.inv[3] * dx + v.inv[4] * dy + v.inv[5] * dz;
  const float qz = v.inv[6] * dx + v.inv[7] * dy + v.inv[8] * dz;
  const float s = fabsf(dx) + fabsf(dy) + fabsf(dz);
  const float iz = __builtin_amdgcn_rcpf(qz);
  const float x = v.fx * qx * iz, y = v.fy * qy * iz;
  float4 r;
  r.x = x + v.cx;
  r.y = y + v.cy;
  r.z = qz;
  r.w = v.rt_abs + (v.rt_rel * s * iz + 9.5367431640625e-07f) * (v.rt_f + fabsf(x) + fabsf(y));
  if (!(qz >= s * 0.015625f && r.w < 1e6f)) r.w = -1.0f;
  return r;
}

// True when every point of the face lies outside one side of the image's
// frustum (a pixel wider than the image on each side, minus the error of q),
// or behind the camera: no ray of the view can hit it. Nor can one hit a face with
// a corner that is not finite: its hit distances are NaN. For faces with a corner
// that project_ray gives no bound for.
UGU_DEV bool outside_frustum(const DevView& v, const float* P) {
  float sum = 0.0f;  // 0 x inf and NaN propagate
  for (int k = 0; k < 9; k++) sum += 0.0f * P[k];
  if (sum != sum) return true;
  int out = 31;
  for (int k = 0; k < 3; k++) {
    const float dx = P[3 * k] - v.c2w_t[0], dy = P[3 * k + 1] - v.c2w_t[1],
                dz = P[3 * k + 2] - v.c2w_t[2];
    const float qx = v.inv[0] * dx + v.inv[1] * dy + v.inv[2] * dz;
    const float qy = v.inv[3] * dx + v.inv[4] * dy + v.inv[5] * dz;
    const float qz = v.inv[6] * dx + v.inv[7] * dy + v.inv[8] * dz;
    const float s = (fabsf(dx) + fabsf(dy) + fabsf(dz)) * (v.rt_rel + 9.5367431640625e-07f);
    const float gx = v.fx * qx, gy = v.fy * qy;
    // pixel x times q.z, against x = -1 and x = W; likewise y
    const float ex = s * (v.rt_f + fabsf(v.cx) + static_cast<float>(v.W) + 1.0f);
    const float ey = s * (v.rt_f + fabsf(v.cy) + static_cast<float>(v.H) + 1.0f);
    int o = 0;
    if (gx + (v.cx + 1.0f) * qz < -ex) o |= 1;
    if (gx + (v.cx - static_cast<float>(v.W)) * qz > ex) o |= 2;
    if (gy + (v.cy + 1.0f) * qz < -ey) o |= 4;
    if (gy + (v.cy - static_cast<float>(v.H)) * qz > ey) o |= 8;
    if (qz < -s) o |= 16;
    out &= o;
  }
  return out != 0;
}

// A bin entry is (face id, depth | box): the upper 16 bits of a float that is
// at most the q.z of every hit of the face (0: no bound), and its pixel box
// within the tile, x | y << 4 | (width - 1) << 8 | (height - 1) << 12.
constexpr int kRtTile = 16;

UGU_DEV int2 rt_entry(int f, float zskip, int x0, int x1, int y0, int y1, int tx, int ty) {
  const int px = tx * kRtTile, py = ty * kRtTile;
  const int lx0 = max(x0 - px, 0), lx1 = min(x1 - px, kRtTile - 1);
  const int ly0 = max(y0 - py, 0), ly1 = min(y1 - py, kRtTile - 1);
  const uint32_t box = lx0 | (ly0 << 4) | ((lx1 - lx0) << 8) | ((ly1 - ly0) << 12);
  return make_int2(f, static_cast<int>((__float_as_uint(zskip) & 0xffff0000u) | box));
}

// One thread per (face, view), as the rasterizer's k_setup_bin: a block's
// distinct vertices are projected once per view into LDS.
// INL: a pass of one view, its descriptor an argument (see k_begin).
template <bool INL>
__global__ __launch_bounds__(256) void k_rt_setup(InlineViews<1> arg,
                                                  const DevView* __restrict__ views, DevView* out,
                                                  int n_views, int block_views, DevMesh mesh,
                                                  DevBins bins, RtLarge large) {
  if (INL && blockIdx.x == 0) {
    // an occupancy published before this store is published again by its tile
    clear_status(bins.status);
    store_inline_views(out, 1);
  }
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int k = threadIdx.x; k < n_views; k += blockDim.x) large.clear[k] = 0;
  __shared__ float4 sp[768];
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  const int vbase = mesh.blk_off[blockIdx.x];
  const int nu = mesh.blk_off[blockIdx.x + 1] - vbase;
  int loc[3] = {0, 0, 0};
  float P[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
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
  const int vb = blockIdx.y * block_views;
  const int ve = min(vb + block_views, n_views);
  for (int vi = vb; vi < ve; vi++) {
    const DevView& v = INL ? arg.v[0] : views[vi];
    for (int j = 0; j < 3; j++) {
      const int k = threadIdx.x + j * 256;
      if (k < nu) sp[k] = project_ray(v, P[j * 3 + 0], P[j * 3 + 1], P[j * 3 + 2]);
    }
    __syncthreads();
    const float4 a = sp[loc[0]], b = sp[loc[1]], c = sp[loc[2]];
    __syncthreads();  // the next view overwrites the window
    bool has = false, back = false;
    float zskip = 0.0f;
    int x0 = 0, x1 = -1, y0 = 0, y1 = -1;
    uint32_t tmask = ~0u;
    if (f < mesh.F) {
      const float zmin = fminf(fminf(a.z, b.z), c.z), zmax = fmaxf(fmaxf(a.z, b.z), c.z);
      // an accepted hit's barycentrics lie within rt_bary of the triangle; on
      // screen that is at most rt_bary zmax / zmin of its extent
      const float rat = v.rt_bary * zmax * __builtin_amdgcn_rcpf(zmin);
      if (fminf(fminf(a.w, b.w), c.w) >= 0.0f && rat < 0.001953125f) {
        const float xl = fminf(fminf(a.x, b.x), c.x), xh = fmaxf(fmaxf(a.x, b.x), c.x);
        const float yl = fminf(fminf(a.y, b.y), c.y), yh = fmaxf(fmaxf(a.y, b.y), c.y);
        const float ext = (xh - xl) + (yh - yl);
        const float w = fmaxf(fmaxf(a.w, b.w), c.w) + 2.0f * rat * ext;
        // |x|, |y| < 1e12 (the bound of w): clamped to the image before the
        // conversion to int
        x0 = static_cast<int>(fmaxf(ceilf(xl - w), 0.0f));
        y0 = static_cast<int>(fmaxf(ceilf(yl - w), 0.0f));
        x1 = static_cast<int>(fminf(floorf(xh + w), static_cast<float>(v.W - 1)));
        y1 = static_cast<int>(fminf(floorf(yh + w), static_cast<float>(v.H - 1)));
        if (!(xl - w <= static_cast<float>(v.W)) || !(yl - w <= static_cast<float>(v.H)) ||
            !(xh + w >= 0.0f) || !(yh + w >= 0.0f)) x1 = -1;
        has = x0 <= x1 && y0 <= y1;
        zskip = zmin * 0.9921875f;
        back = !(edge_fn(a.x, a.y, b.x, b.y, c.x, c.y) > 0.0f);
        if (has && (x1 - x0 + 1) * (y1 - y0 + 1) <= kCoverProbe) {
          // at most 2 x 2 tiles: only those with a pixel centre the face's
          // hits can reach. A corner moved by w moves an edge function at a
          // centre of the box by at most 3 w ext + 4 w w (the box is w wider).
          const float tol = 3.0f * w * (ext + 4.0f * w) + 4.0f * w * w;
          const int tx0 = x0 / kRtTile, ty0 = y0 / kRtTile;
          tmask = 0u;
          int px = x0, py = y0;
#pragma unroll
          for (int k = 0; k < kCoverProbe; k++) {
            if (py <= y1) {
              const float x = static_cast<float>(px), y = static_cast<float>(py);
              const float w0 = edge_fn(b.x, b.y, c.x, c.y, x, y);
              const float w1 = edge_fn(c.x, c.y, a.x, a.y, x, y);
              const float w2 = edge_fn(a.x, a.y, b.x, b.y, x, y);
              if (fminf(fminf(w0, w1), w2) >= -tol || fmaxf(fmaxf(w0, w1), w2) <= tol)
                tmask |= 1u << ((px / kRtTile - tx0) + 2 * (py / kRtTile - ty0));
              if (++px > x1) {
                px = x0;
                py++;
              }
            }
          }
          has = tmask != 0u;
        }
      } else {
        float Q[9];
        const float4* r = mesh.soup + int64_t(f) * 3;
        const float4 r0 = r[0], r1 = r[1], r2 = r[2];
        Q[0] = r0.x; Q[1] = r0.y; Q[2] = r0.z;
        Q[3] = r0.w; Q[4] = r1.x; Q[5] = r1.y;
        Q[6] = r1.z; Q[7] = r1.w; Q[8] = r2.x;
        has = !outside_frustum(v, Q);
        x0 = y0 = 0;
        x1 = v.W - 1;
        y1 = v.H - 1;
      }
    }
    // A large face would be appended to its bins by this wavefront alone, 64 tiles at
    // a time: a ball in a room of 12 faces at 1080p 2330 us, listed 121 (hierarchy
    // 319); 82 k faces seen from close by at 640x480 107 and 78 (81).
    const int tiles = (x1 / kRtTile - x0 / kRtTile + 1) * (y1 / kRtTile - y0 / kRtTile + 1);
    const uint64_t big = __builtin_amdgcn_ballot_w64(
        has && tiles > max(kRtLargeTiles, v.tiles_x * v.tiles_y / kRtLargeShare));
    if (big) {
      const int lane = __lane_id(), lead = __ffsll(static_cast<unsigned long long>(big)) - 1;
      int slot = 0;
      if (lane == lead) slot = atomicAdd(&large.count[vi], __popcll(big));
      slot = __shfl(slot, lead) + __popcll(big & ((1ull << lane) - 1ull));
      if (((big >> lane) & 1ull) && slot < kRtLargeFaces) {
        large.list[int64_t(vi) * kRtLargeFaces + slot] =
            make_int4(f, __float_as_int(zskip), x0 | (x1 << 16), y0 | (y1 << 16));
        has = false;
      }
    }
    const int tx0 = x0 / kRtTile, tx1 = has ? x1 / kRtTile : -1;
    const int ty0 = y0 / kRtTile, ty1 = has ? y1 / kRtTile : -1;
    const uint32_t zmin = back_zmin(has && back, __uint_as_float(__float_as_uint(zskip) & 0xffff0000u));
    const int nx = tx1 - tx0 + 1;
    const int rest = has ? max(nx * (ty1 - ty0 + 1) - kAppendRounds, 0) : 0;
    int tx = tx0, ty = ty0;
    const bool probed = tmask != ~0u;
    uint32_t pm = tmask;
    AppendTicket tk[kAppendRounds];
    int2 entry[kAppendRounds];
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
      entry[r] = rt_entry(f, zskip, x0, x1, y0, y1, ax, ay);
      tk[r] = append_issue(bins, has ? 4 * (v.tile_base + ay * v.tiles_x + ax) + (back ? 1 : 0) : -1,
                           zmin, has);
      if (probed) {
        pm &= pm - 1u;
        has = has && pm != 0u;
      } else if (has && ++tx > tx1) {
        tx = tx0;
        if (++ty > ty1) has = false;
      }
    }
    append_finish<kAppendRounds, true>(bins, tk, entry, used);
    // faces over more tiles: 64 (face, tile) pairs of the wavefront at a time
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
        const int snx = max(__shfl(nx, src), 1);
        const int sx0 = __shfl(x0, src), sx1 = __shfl(x1, src);
        const int sy0 = __shfl(y0, src), sy1 = __shfl(y1, src);
        const int sty = sy0 / kRtTile + k / snx;
        const int stx = sx0 / kRtTile + k % snx;
        const int sback = __shfl(back ? 1 : 0, src);
        const int2 e = rt_entry(__shfl(f, src), __shfl(zskip, src), sx0, sx1, sy0, sy1, stx, sty);
        // mostly different tiles, so every lane appends its own (grouped by tile as in
        // append_issue: 10 k faces of 100 tiles at 1080p 857 us, so 429)
        if (p < total) {
          const int tile = v.tile_base + sty * v.tiles_x + stx;
          const int slot = atomicAdd(&bins.counts[4 * tile + sback], 1);
          if (sback) atomicMin(reinterpret_cast<unsigned int*>(bins.counts) + (4 * tile + 2), zmin);
          if (slot < bins.cap)
            bins.bins[int64_t(tile) * bins.cap + (sback ? bins.cap - 1 - slot : slot)] = e;
          else
            atomicMax(&bins.status[0], slot + 1);
        }
      }
    }
  }
}

struct RtLds {
  unsigned long long key[256];  // packed (hit distance bits << 32 | face id)
  float ray[3][256];            // ray_w of each tile pixel
  float p[9][256];              // staged faces: corner positions
  int32_t fid[256];
  uint16_t box[256];            // rt_entry's pixel box
  PairLds<256> pairs;
  uint32_t wmax[4];
};

// One 16 x 16 pixel tile: its bin's faces are staged 256 at a time, expanded
// to (face, pixel) pairs (as raster_tile does) and every pair runs the float64
// hit test; a pixel keeps its smallest (distance, face id) with one LDS
// atomicMin. Faces whose depth bound lies behind every hit of the tile are
// dropped before their positions are fetched: the tile's bound is the largest
// q.z = distance * (z of the normalized camera-space ray) its pixels hold, and a
// face with all its q.z beyond it (by more than 2^-8, far above the float32
// rounding of either) is hit later than what each pixel holds.
// Bound by the latency of a tile's dependent loads (counters, entries, face
// records, the winner's record and shading inputs), like k_raster. 1.3 M faces
// at 1080p: setup 27 us + tiles 53 us, where the hierarchy walk (k_raytrace)
// takes 836 us; 24 mixed views of 492 k faces: 153 + 295 us against 2505 us. 6
// waves per SIMD (78 VGPRs, the rays in LDS only): 5 take 330 us, 7 spill, 333 us.
__global__ __launch_bounds__(256, 6) void k_rt_tiles(const DevView* __restrict__ views, DevMesh m,
                                                  DevBins bins, RtLarge large, DevOptions o) {
  constexpr int NT = 256;
  __shared__ RtLds s;
  const int t = threadIdx.x;
  const int gtile = xcd_remap(blockIdx.x, gridDim.x);
  const int4 seg = reinterpret_cast<const int4*>(bins.counts)[gtile];
  // Some bin overflowed: the host renders again, nothing here is worth finishing.
  // Both conditions are the same in every thread of the block: status[0] is the
  // setup kernel's and no block writes it here (a word that blocks of this launch
  // raise would let a block's wavefronts differ, and those that stay read LDS that
  // the leavers never wrote). A tile that its two segments overflow together is
  // first seen here, and published in status[1].
  if (seg.x + seg.y > bins.cap || bins.status[0] > bins.cap) {
    if (t == 0 && seg.x + seg.y > bins.cap) {
      atomicMax(&bins.status[1], seg.x + seg.y);
      *bins.host_flag = 1;
    }
    return;
  }
  const DevView& v = views[seg.w];
  const int lt = gtile - v.tile_base;
  const int tyi = lt / v.tiles_x, txi = lt - tyi * v.tiles_x;
  const int gx = txi * kRtTile + t % kRtTile, gy = tyi * kRtTile + t / kRtTile;
  const bool act = gx < v.W && gy < v.H;
  const int nA = seg.x, nB = seg.y, n = nA + nB;
  const int n_large = min(large.count[seg.w], kRtLargeFaces);
  int bf = -1;
  float r0 = 0.0f, r1 = 0.0f, r2 = 0.0f;
  if (n + n_large > 0) {
    const int2* bin = bins.bins + int64_t(gtile) * bins.cap;
    const int4* list = large.list + int64_t(seg.w) * kRtLargeFaces;
    // chunks of 256 faces: of the view's large faces (ch < 0), of the bin's front
    // and of its back segment
    const int chunks_l = (n_large + NT - 1) / NT;
    const int chunks_a = (nA + NT - 1) / NT, chunks = chunks_a + (nB + NT - 1) / NT;
    int2 e_next = make_int2(0, 0);
    if (t < (chunks_a > 0 ? nA : n)) e_next = bin_entry(bin, nA, bins.cap, t);
    {
      float w0, w1, w2;
      ray_w_at(v, static_cast<float>(gx), static_cast<float>(gy), w0, w1, w2);
      s.ray[0][t] = w0;
      s.ray[1][t] = w1;
      s.ray[2][t] = w2;
    }
    // z of the pixel's normalized camera-space ray: q.z of a hit at distance 1
    const float u0 = (static_cast<float>(gx) - v.cx) / v.fx;
    const float u1 = (static_cast<float>(gy) - v.cy) / v.fy;
    const float zray = __builtin_amdgcn_rsqf(u0 * u0 + u1 * u1 + 1.0f);
    const double ox = v.c2w_t[0], oy = v.c2w_t[1], oz = v.c2w_t[2];
    s.key[t] = ~0ull;
    float dmax = __uint_as_float(0xffffffffu);  // NaN: some pixel has no hit yet
    for (int ch = -chunks_l; ch < chunks; ch++) {
      if (ch == chunks_a && skip_face(__uint_as_float(static_cast<uint32_t>(seg.z)), dmax)) break;
      int base = ch < chunks_a ? ch * NT : nA + (ch - chunks_a) * NT;
      int end = ch < chunks_a ? nA : n;
      const bool more = ch + 1 < chunks;
      int2 e = e_next;
      if (ch < 0) {
        base = (ch + chunks_l) * NT;
        end = 0;  // unless the face's box meets the tile
        if (base + t < n_large) {
          const int4 q = list[base + t];
          const int x0 = q.z & 0xffff, x1 = static_cast<uint32_t>(q.z) >> 16;
          const int y0 = q.w & 0xffff, y1 = static_cast<uint32_t>(q.w) >> 16;
          if (x0 < (txi + 1) * kRtTile && x1 >= txi * kRtTile && y0 < (tyi + 1) * kRtTile &&
              y1 >= tyi * kRtTile) {
            e = rt_entry(q.x, __int_as_float(q.y), x0, x1, y0, y1, txi, tyi);
            end = n_large;
          }
        }
      } else if (more) {
        const int nbase = ch + 1 < chunks_a ? (ch + 1) * NT : nA + (ch + 1 - chunks_a) * NT;
        const int nend = ch + 1 < chunks_a ? nA : n;
        e_next = nbase + t < nend ? bin_entry(bin, nA, bins.cap, nbase + t) : make_int2(0, 0);
      }
      int c = 0;
      if (base + t < end &&
          !skip_face(__uint_as_float(static_cast<uint32_t>(e.y) & 0xffff0000u), dmax)) {
        const float4* r = m.soup + int64_t(e.x) * 3;
        const float4 a = r[0], b = r[1], d = r[2];
        s.p[0][t] = a.x; s.p[1][t] = a.y; s.p[2][t] = a.z;
        s.p[3][t] = a.w; s.p[4][t] = b.x; s.p[5][t] = b.y;
        s.p[6][t] = b.z; s.p[7][t] = b.w; s.p[8][t] = d.x;
        s.fid[t] = e.x;
        s.box[t] = static_cast<uint16_t>(e.y);
        c = (((e.y >> 8) & 15) + 1) * (((e.y >> 12) & 15) + 1);
      }
      const int lane = t & 63, wid = t >> 6;
      publish_pairs(s.pairs, ch & 1, c);
      __syncthreads();
      auto test_pair = [&](int j, int pix) {
        const float3 p0 = make_float3(s.p[0][j], s.p[1][j], s.p[2][j]);
        const float3 p1 = make_float3(s.p[3][j], s.p[4][j], s.p[5][j]);
        const float3 p2 = make_float3(s.p[6][j], s.p[7][j], s.p[8][j]);
        float ht, hu, hv;
        if (mt_hit(ox, oy, oz, s.ray[0][pix], s.ray[1][pix], s.ray[2][pix], p0, p1, p2, ht, hu,
                   hv) &&
            ht < __builtin_huge_valf()) {
          // + 0: a distance of -0 becomes 0, so the bits order as the floats
          const unsigned long long key =
              (static_cast<unsigned long long>(__float_as_uint(ht + 0.0f)) << 32) |
              static_cast<unsigned int>(s.fid[j]);
          atomicMin(&s.key[pix], key);
        }
      };
      auto locate = [&](int j, int r, int& pix) {
        const int bx = s.box[j];
        const int nx = ((bx >> 8) & 15) + 1;
        const int qy = pair_row(r, nx);
        pix = (((bx >> 4) & 15) + qy) * kRtTile + (bx & 15) + (r - qy * nx);
        return true;
      };
      if (walk_pairs<NT, true>(s.pairs, ch & 1, locate, test_pair) == 0) continue;
      __syncthreads();
      if (more) {
        const unsigned long long k = s.key[t];
        // depth of the pixel's hit: all ones when it has none, 0 outside the image
        uint32_t db = 0u;
        if (act) {
          const uint32_t tb = static_cast<uint32_t>(k >> 32);
          db = k == ~0ull ? 0xffffffffu : __float_as_uint(__uint_as_float(tb) * zray);
        }
        db = wave_max_u32(db);
        if (lane == 0) s.wmax[wid] = db;
        __syncthreads();
        uint32_t mx = s.wmax[0];
        for (int w = 1; w < NT / 64; w++) mx = max(mx, s.wmax[w]);
        dmax = __uint_as_float(mx);
      }
    }
    const unsigned long long k = s.key[t];
    if (k != ~0ull) bf = static_cast<int>(static_cast<unsigned int>(k & 0xffffffffull));
    r0 = s.ray[0][t];
    r1 = s.ray[1][t];
    r2 = s.ray[2][t];
  }
  if (!act) return;
  float bt = 0.0f, bu = 0.0f, bv = 0.0f;
  if (bf >= 0) {
    // the winner's distance and weights, by the test that accepted it
    const float4* r = m.soup + int64_t(bf) * 3;
    const float4 a = r[0], b = r[1], d = r[2];
    const float3 p0 = make_float3(a.x, a.y, a.z), p1 = make_float3(a.w, b.x, b.y),
                 p2 = make_float3(b.z, b.w, d.x);
    mt_hit(v.c2w_t[0], v.c2w_t[1], v.c2w_t[2], r0, r1, r2, p0, p1, p2, bt, bu, bv);
  }
  write_hit<true>(v, m, o, gx, gy, bf, bt, bu, bv, r0, r1, r2);
  // the tile's counters, cleared for the next pass (see raster_tile)
  if (t == 0 && n > 0)
    reinterpret_cast<int4*>(bins.counts)[gtile] = make_int4(0, 0, 0x7f800000, seg.w);
}

// ---------------------------------------------------------------------------
// Visibility test: VisibilityTester::TestVertex (visibility_tester.cc:390-530)
// for one item per lane. Items are scattered over the image, so every lane
// walks the hierarchy on its own (stack of kBvhStack entries per lane in LDS).

struct DevVisItem {
  int32_t visible;
  float px, py, angle, dist, c0, c1, c2, intensity;
};

// closest float t over all faces (+inf: no hit), per-lane traversal
UGU_DEV float closest_t(const BvhNode* __restrict__ nodes, const int2* __restrict__ leaves,
                        const float4* __restrict__ tris, int32_t* stack, int lane, float ox,
                        float oy, float oz, float r0, float r1, float r2) {
  const float ix = 1.0f / r0, iy = 1.0f / r1, iz = 1.0f / r2;
  const double dox = ox, doy = oy, doz = oz;
  float bt = __builtin_huge_valf();
  float tmax = bt;  // box_tmax(bt), updated with bt
  int sp = 0, ref = 0;
  for (;;) {
    if (ref >= 0) {
      const BvhNode nd = nodes[ref];
      const int ra = __float_as_int(nd.a_lo.w), rb = __float_as_int(nd.b_lo.w);
      const float ta = box_entry(nd.a_lo, nd.a_hi, ox, oy, oz, ix, iy, iz, tmax);
      const float tb = rb == kBvhEmpty ? __builtin_huge_valf()
                                       : box_entry(nd.b_lo, nd.b_hi, ox, oy, oz, ix, iy, iz, tmax);
      const bool ha = ta != __builtin_huge_valf(), hb = tb != __builtin_huge_valf();
      if (ha && hb) {
        const bool a_first = ta <= tb;
        stack[sp * 64 + lane] = a_first ? rb : ra;
        sp++;
        ref = a_first ? ra : rb;
        continue;
      }
      if (ha || hb) {
        ref = ha ? ra : rb;
        continue;
      }
    } else {
      const int2 lf = leaves[~ref];
      for (int k = 0; k < lf.y; k++) {
        const float4* tr = tris + int64_t(lf.x + k) * 3;
        float t, u, w;
        if (mt_hit(dox, doy, doz, r0, r1, r2, tr[0], tr[1], tr[2], t, u, w) && t < bt) {
          bt = t;
          tmax = box_tmax(bt);
        }
      }
    }
    if (sp == 0) break;
    sp--;
    ref = stack[sp * 64 + lane];
  }
  return bt;
}

__global__ __launch_bounds__(64) void k_visibility(DevView v, const uint8_t* __restrict__ color,
                                                   const float* __restrict__ depth,
                                                   const uint8_t* __restrict__ mask,
                                                   DevVisOpt o, int n,
                                                   const float* __restrict__ pos,
                                                   const float* __restrict__ vert,
                                                   const float* __restrict__ nrm,
                                                   const BvhNode* __restrict__ nodes,
                                                   const int2* __restrict__ leaves,
                                                   const float4* __restrict__ tris,
                                                   DevVisItem* __restrict__ out) {
  __shared__ int32_t stack[kBvhStack * 64];
  const int lane = threadIdx.x;
  const int i = blockIdx.x * 64 + lane;
  if (i >= n) return;
  DevVisItem r;
  r.visible = 0;
  r.px = r.py = r.c0 = r.c1 = r.c2 = 0.0f;
  r.angle = 999.9f;
  r.dist = -999.9f;
  r.intensity = -1.0f;
  const float px = pos[i * 3], py = pos[i * 3 + 1], pz = pos[i * 3 + 2];
  // camera_p = w2c * world_p, then Project(camera_p, &image_p, &d)
  const float qx = sum3(v.w2c_R[0] * px, v.w2c_R[1] * py, v.w2c_R[2] * pz) + v.w2c_t[0];
  const float qy = sum3(v.w2c_R[3] * px, v.w2c_R[4] * py, v.w2c_R[5] * pz) + v.w2c_t[1];
  const float qz = sum3(v.w2c_R[6] * px, v.w2c_R[7] * py, v.w2c_R[8] * pz) + v.w2c_t[2];
  const float ix = v.fx / qz * qx + v.cx;
  const float iy = v.fy / qz * qy + v.cy;
  for (;;) {  // one pass; `break` = TestVertex returns false
    if (qz < 0.0f || ix < 0.0f || static_cast<float>(v.W - 1) < ix || iy < 0.0f ||
        static_cast<float>(v.H - 1) < iy)
      break;
    if (!(ix >= 0.0f && iy >= 0.0f)) break;  // NaN projections
    const int nx = static_cast<int>(roundf(ix)), ny = static_cast<int>(roundf(iy));
    const int64_t pi = int64_t(ny) * v.W + nx;
    if (o.use_mask && mask[pi] != 255) break;
    if (o.use_depth && depth[pi] < FLT_EPSILON) break;
    float r0, r1, r2;
    ray_w_at(v, ix, iy, r0, r1, r2);
    const float dot = -sum3(nrm[i * 3] * r0, nrm[i * 3 + 1] * r1, nrm[i * 3 + 2] * r2);
    const float angle = acosf(dot);
    if (o.th < angle) break;
    const float ox = v.c2w_t[0], oy = v.c2w_t[1], oz = v.c2w_t[2];
    const float t = closest_t(nodes, leaves, tris, stack, lane, ox, oy, oz, r0, r1, r2);
    const float vx = vert[i * 3], vy = vert[i * 3 + 1], vz = vert[i * 3 + 2];
    float hx = vx, hy = vy, hz = vz;
    const float distance = t < __builtin_huge_valf() ? t : FLT_MAX;
    if (t < __builtin_huge_valf()) {
      hx = ox + r0 * t;
      hy = oy + r1 * t;
      hz = oz + r2 * t;
      const float dx = hx - vx, dy = hy - vy, dz = hz - vz;
      if (sqrtf(sum3(dx * dx, dy * dy, dz * dz)) > o.eps) break;
    }
    if (o.use_depth) {
      const float hcz = sum3(v.w2c_R[6] * hx, v.w2c_R[7] * hy, v.w2c_R[8] * hz) + v.w2c_t[2];
      if (o.max_ddiff < fabsf(hcz - depth[pi])) break;
    }
    r.px = ix;
    r.py = iy;
    r.angle = angle;
    r.dist = distance;
    if (distance > o.max_dist || angle > o.max_angle) break;
    float c[3];
    if (o.interp == 0) {
      for (int k = 0; k < 3; k++) c[k] = static_cast<float>(color[pi * 3 + k]);
    } else {
      // BilinearInterpolation (include/ugu/util/image_util.h:155-193)
      int x0 = static_cast<int>(floorf(ix)), y0 = static_cast<int>(floorf(iy));
      int x1 = x0 + 1, y1 = y0 + 1;
      if (x0 < 0) x0 = 0;
      if (y0 < 0) y0 = 0;
      if (v.W <= x1) x1 = v.W - 1;
      if (v.H <= y1) y1 = v.H - 1;
      const float lu = ix - static_cast<float>(x0), lv = iy - static_cast<float>(y0);
      const uint8_t* c00 = color + (int64_t(y0) * v.W + x0) * 3;
      const uint8_t* c01 = color + (int64_t(y0) * v.W + x1) * 3;
      const uint8_t* c10 = color + (int64_t(y1) * v.W + x0) * 3;
      const uint8_t* c11 = color + (int64_t(y1) * v.W + x1) * 3;
      for (int k = 0; k < 3; k++) {
        const float f = (1.0f - lu) * (1.0f - lv) * static_cast<float>(c00[k]) +
                        lu * (1.0f - lv) * static_cast<float>(c01[k]) +
                        (1.0f - lu) * lv * static_cast<float>(c10[k]) +
                        lu * lv * static_cast<float>(c11[k]);
        c[k] = static_cast<float>(f2u8_x86(f));
      }
    }
    r.c0 = c[0];
    r.c1 = c[1];
    r.c2 = c[2];
    // Color2Gray (image_util.h:227-244): double arithmetic, cast to float
    r.intensity = static_cast<float>(0.2989 * double(c[0]) + 0.5870 * double(c[1]) +
                                     0.1140 * double(c[2]));
    r.visible = 1;
    break;
  }
  out[i] = r;
}

int launch_visibility(hipStream_t st, const DevView& v, const uint8_t* color, const float* depth,
                      const uint8_t* mask, const DevVisOpt& o, int n, const float* pos,
                      const float* vert, const float* nrm, const DevBvh& bvh, void* out) {
  if (n < 1) return 0;
  hipLaunchKernelGGL(k_visibility, dim3((n + 63) / 64), dim3(64), 0, st, v, color, depth, mask, o,
                     n, pos, vert, nrm, bvh.nodes, bvh.leaves, bvh.tris,
                     static_cast<DevVisItem*>(out));
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// views[i].tile_base = first 16x16 tile of view i; the bins' counters cleared.
// one: as launch_setup_bin's
int launch_raytrace_binned(hipStream_t st, const DevView* one, DevView* views, int n_views,
                           const DevMesh& m, const DevBins& bins, const RtLarge& large,
                           const DevOptions& o) {
  if (n_views < 1 || bins.total_tiles < 1 || m.F < 1) return 0;
  // a block's faces stay for kSetupViews views, fewer where the blocks would not fill
  // the chip (320 faces, 24 views of 640x480: 661 us with eight,
  // 550 with one)
  const int fb = (m.F + 255) / 256;
  const int per = std::max(1, std::min<int>(kSetupViews, int64_t(fb) * n_views / 1024));
  const dim3 grid(fb, (n_views + per - 1) / per);
  InlineViews<1> a{};
  if (one) {
    a.v[0] = *one;
    hipLaunchKernelGGL(k_rt_setup<true>, grid, dim3(256), 0, st, a, nullptr, views, 1, 1, m, bins,
                       large);
  } else {
    hipLaunchKernelGGL(k_rt_setup<false>, grid, dim3(256), 0, st, a, views, nullptr, n_views, per, m,
                       bins, large);
  }
  hipLaunchKernelGGL(k_rt_tiles, dim3(bins.total_tiles), dim3(256), 0, st, views, m, bins, large,
                     o);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// views[i].tile_base = first 8x8 tile of view i in the concatenated tile list
int launch_raytrace(hipStream_t st, const DevView* views, int n_views, int total_tiles,
                    const DevBvh& bvh, const DevMesh& m, const DevOptions& o) {
  if (n_views < 1 || total_tiles < 1) return 0;
  // One view: each XCD takes one contiguous band of tiles (measured 0.61 vs
  // 0.75 ms at 1080p). Many views: runs of 16 workgroups alternate over the
  // XCDs (views differ in cost per tile; one band per XCD would leave some
  // XCDs with the expensive views: 13.8 vs 10.5 ms on the 64 ring views).
  const int64_t need = (int64_t(total_tiles) + kRtWaves - 1) / kRtWaves;
  const int64_t chunk = n_views == 1 ? (need + 7) / 8 : 16;
  const int64_t per = 8 * chunk;
  const int64_t blocks64 = (need + per - 1) / per * per;
  if (blocks64 > INT32_MAX) return -1;
  const int blocks = static_cast<int>(blocks64);
  hipLaunchKernelGGL(k_raytrace, dim3(blocks), dim3(64 * kRtWaves), 0, st, views, bvh.nodes,
                     bvh.leaves, bvh.tris, n_views, total_tiles, static_cast<int>(chunk), m, o);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugu_hip
