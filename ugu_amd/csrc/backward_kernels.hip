// Differentiable backward pass (no reference counterpart): dL/d(vertices,
// vertex colours, texture) at fixed visibility. The covered pixels of all views
// are sorted into (face, view, pixel) items by groups of consecutive faces with
// a counting sort:
//   k_bwd_count    four pixels per thread: pixels per face group
//   k_bwd_offsets  exclusive scan of the counts (one launch, at most 16 blocks, each
//                  of which sums the counts before its own)
//   k_bwd_scatter  four pixels per thread: the items
//   k_bwd_items    one thread per item: derivatives in float64, summed per
//                  vertex and texel in a block's LDS tables before the global
//                  atomics
// A block's consecutive items are the pixels, in every view, of a few
// neighbouring faces, so its contributions meet at few vertices and texels; and
// the items of one group in one view are runs of neighbouring pixels, so the
// gradient image is read in runs too.

#include "device_common.h"

#pragma clang fp contract(off)

namespace ugu_hip {

// Faces fid >> shift share a group; the shift keeps the groups below kBwdGroups.
// Coarse groups give long runs: 64 views of 1.3 M faces take 0.5 M counter atomics
// per pass instead of 6.8 M with a counter per face (count 281 -> 130 us, scatter
// 404 -> 166 us), and the offsets fit one kernel instead of three.
constexpr int kBwdGroups = 16384;

int backward_group_shift(int32_t F) {
  int shift = 0;
  while (((F - 1) >> shift) >= kBwdGroups) shift++;
  return shift;
}

// A wavefront's 8x8 pixel square and its pixels' face groups. Each pass of the
// loop takes the lowest lane not grouped yet; the lanes with its group form one
// set, led by that lane. rank: the lane's place in its set.
struct GroupSet {
  uint64_t mask;
  int rank, leader;
};

UGU_DEV GroupSet group_lanes(int group, bool valid) {
  GroupSet g;
  g.mask = 0;
  const uint64_t all = __builtin_amdgcn_ballot_w64(valid);
  uint64_t todo = all;
  while (todo) {
    const int l = __ffsll(static_cast<unsigned long long>(todo)) - 1;
    const int lg = __builtin_amdgcn_readlane(group, l);
    const uint64_t set = __builtin_amdgcn_ballot_w64(group == lg) & all;
    g.mask = (valid && group == lg) ? set : g.mask;
    todo &= ~set;
  }
  g.rank = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
      static_cast<uint32_t>(g.mask >> 32),
      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(g.mask), 0u)));
  g.leader = valid ? __ffsll(static_cast<unsigned long long>(g.mask)) - 1 : 0;
  return g;
}

// A block's pixels: kBwdSquares neighbouring squares of 16 x 16 pixels of view
// blockIdx.y, one of each per thread; a wavefront has an 8 x 8 square of them.
// The face ids are read together, so a thread waits for one round trip. 0: no
// face to count (face 0 is never shaded, rasterizer.cc:250, so it has no
// gradient).
constexpr int kBwdSquares = 4;

struct BwdPixels {
  int fid[kBwdSquares];
  int x[kBwdSquares], y[kBwdSquares];
};

UGU_DEV void bwd_pixels(const DevView& v, int32_t F, BwdPixels& p) {
  const int sw = (v.W + 15) >> 4;
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const int lx = (wid & 1) * 8 + (lane & 7), ly = (wid >> 1) * 8 + (lane >> 3);
  for (int k = 0; k < kBwdSquares; k++) {
    const int sq = static_cast<int>(blockIdx.x) * kBwdSquares + k;
    p.y[k] = sq / sw * 16 + ly;
    p.x[k] = sq % sw * 16 + lx;
    p.fid[k] = (p.x[k] < v.W && p.y[k] < v.H) ? v.face_id[int64_t(p.y[k]) * v.W + p.x[k]] : 0;
  }
  for (int k = 0; k < kBwdSquares; k++)
    if (!(p.fid[k] > 0 && p.fid[k] < F)) p.fid[k] = 0;
}

__global__ __launch_bounds__(256) void k_bwd_count(const DevView* __restrict__ views, int32_t F,
                                                   int shift, int32_t* __restrict__ cnt) {
  BwdPixels p;
  bwd_pixels(views[blockIdx.y], F, p);
  for (int k = 0; k < kBwdSquares; k++) {
    const GroupSet g = group_lanes(p.fid[k] >> shift, p.fid[k] > 0);
    if (p.fid[k] > 0 && g.rank == 0) atomicAdd(&cnt[p.fid[k] >> shift], __popcll(g.mask));
  }
}

// Exclusive scan of n <= kBwdGroups counts into `cursor` (its entry n gets the
// total): block b sums the counts before its 1024 and scans its own.
__global__ __launch_bounds__(1024) void k_bwd_offsets(const int32_t* __restrict__ cnt, int n,
                                                      int32_t* __restrict__ cursor) {
  __shared__ int32_t wsum[2][16];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  const int i = static_cast<int>(blockIdx.x) * 1024 + t;
  int before = 0;
  for (int k = 0; k < static_cast<int>(blockIdx.x); k++) before += cnt[k * 1024 + t];
  const int v = i < n ? cnt[i] : 0;
  const int x = wave_incl_sum(v), y = wave_incl_sum(before);
  if (lane == 63) {
    wsum[0][wid] = x;
    wsum[1][wid] = y;
  }
  __syncthreads();
  int base = x - v;
  for (int w = 0; w < 16; w++) base += wsum[1][w] + (w < wid ? wsum[0][w] : 0);
  if (i < n) cursor[i] = base;
  if (i == n - 1) cursor[n] = base + v;
}

// Writes the items, each group's from its cursor on, and clears the counts for
// the next call.
__global__ __launch_bounds__(256) void k_bwd_scatter(const DevView* __restrict__ views, int32_t F,
                                                     int shift, int32_t* __restrict__ cnt,
                                                     int32_t* __restrict__ cursor,
                                                     int4* __restrict__ items) {
  const int blocks = gridDim.x * gridDim.y, b = blockIdx.y * gridDim.x + blockIdx.x;
  for (int i = b * 256 + threadIdx.x; i < kBwdGroups; i += blocks * 256) cnt[i] = 0;
  const DevView& v = views[blockIdx.y];
  BwdPixels p;
  bwd_pixels(v, F, p);
  GroupSet g[kBwdSquares];
  int base[kBwdSquares];
  for (int k = 0; k < kBwdSquares; k++) {
    g[k] = group_lanes(p.fid[k] >> shift, p.fid[k] > 0);
    base[k] = 0;
    if (p.fid[k] > 0 && g[k].rank == 0)
      base[k] = atomicAdd(&cursor[p.fid[k] >> shift], __popcll(g[k].mask));
  }
  for (int k = 0; k < kBwdSquares; k++) {
    const int at = __shfl(base[k], g[k].leader) + g[k].rank;
    if (p.fid[k] > 0)
      items[at] = make_int4(p.fid[k], blockIdx.y, p.x[k] | (p.y[k] << 16), p.y[k] * v.W + p.x[k]);
  }
}

// ---------------------------------------------------------------------------

// LDS tables of a block, open addressing: texels (3 sums) and vertices (3
// position and 3 colour sums). Contributions that find no slot go straight to
// global atomics. The sums are float64: an LDS atomic add of a float64 takes 13 to
// 37 cycles of the CU per wavefront (no, some, many equal addresses), one of a
// float32 194 whatever the addresses.
constexpr int kBwdThreads = 512;
constexpr int kTexProbes = 8;
constexpr int kVtxProbes = 6;
constexpr int kBwdCams = 64;  // views whose cameras are kept in LDS

// Camera of an item's view: in LDS as float64 (at most kBwdCams views), or read
// from the view descriptor.
struct BwdCam {
  double fx, fy, cx, cy;
  double R[9], t[3];
  const float* grad;
};

template <bool LDS>
struct CamRef;

template <>
struct CamRef<true> {
  const BwdCam& c;
  UGU_DEV CamRef(const BwdCam* lds, const DevView*, int i) : c(lds[i]) {}
  UGU_DEV double fx() const { return c.fx; }
  UGU_DEV double fy() const { return c.fy; }
  UGU_DEV double cx() const { return c.cx; }
  UGU_DEV double cy() const { return c.cy; }
  UGU_DEV double R(int k) const { return c.R[k]; }
  UGU_DEV double t(int k) const { return c.t[k]; }
  UGU_DEV const float* grad() const { return c.grad; }
};

template <>
struct CamRef<false> {
  const DevView& v;
  UGU_DEV CamRef(const BwdCam*, const DevView* views, int i) : v(views[i]) {}
  UGU_DEV double fx() const { return v.fx; }
  UGU_DEV double fy() const { return v.fy; }
  UGU_DEV double cx() const { return v.cx; }
  UGU_DEV double cy() const { return v.cy; }
  UGU_DEV double R(int k) const { return v.w2c_R[k]; }
  UGU_DEV double t(int k) const { return v.w2c_t[k]; }
  UGU_DEV const float* grad() const { return v.grad; }
};

// Slots by what the pass learns: two blocks of either fit the 160 KB of a CU.
template <bool TEX, bool VTX>
struct BwdLds {
  static constexpr int kTex = !TEX ? 16 : VTX ? 1792 : 2528;  // multiples of 4
  static constexpr int kVtx = !VTX ? 4 : TEX ? 384 : 1024;
  double tval[3][kTex];
  double vval[6][kVtx];
  BwdCam cam[kBwdCams];
  int32_t tkey[kTex];
  int32_t vkey[kVtx];
};

// First slot of a texel: four neighbouring texels of a row take neighbouring
// slots, so that the flush writes them together; the quadruples are spread.
template <int SLOTS>
UGU_DEV int tex_slot(int x, int y) {
  const uint32_t h = (static_cast<uint32_t>(x) >> 2) * 2654435761u + static_cast<uint32_t>(y) * 2246822519u;
  return static_cast<int>(__umulhi(h ^ (h << 15), SLOTS / 4) * 4) + (x & 3);
}

// Slot of `key`, taking a free one; -1 when the probed ones hold other keys.
template <int SLOTS, int STEP, int PROBES>
UGU_DEV int find_slot(int32_t* keys, int h, int key) {
  static_assert(STEP < SLOTS, "one wrap per step");
#pragma unroll 1
  for (int p = 0; p < PROBES; p++) {
    const int old = atomicCAS(&keys[h], -1, key);
    if (old == -1 || old == key) return h;
    h += STEP;
    if (h >= SLOTS) h -= SLOTS;
  }
  return -1;
}

// Adds 9 values (3 per corner) to the LDS sums of their corners' vertices.
template <int N>
UGU_DEV void add_corners(double (*sum)[N], const int* slot, const int* vid, const float* val,
                         float* __restrict__ global) {
  for (int i = 0; i < 3; i++) {
    if (slot[i] >= 0) {
      for (int k = 0; k < 3; k++) unsafeAtomicAdd(&sum[k][slot[i]], double(val[3 * i + k]));
    } else {
      for (int k = 0; k < 3; k++)
        unsafeAtomicAdd(&global[int64_t(vid[i]) * 3 + k], val[3 * i + k]);
    }
  }
}

// One thread per item, `rounds` items each; a block's items are consecutive.
//
// Geometry at the pixel, with the corners' screen positions relative to it
// (X', Y'): the edge functions are e0 = X2' Y1' - X1' Y2' and so on, the weights
// b_i = q_i / (q0 + q1 + q2) with q_i = e_i / Z_i (the triangle's area cancels).
// With G_j = dL/db_j - sum_i dL/db_i b_i: dL/de_j = G_j / (Z_j sum q),
// dL/dZ_j = -G_j b_j / Z_j + the terms through X, Y.
//
// 4 wavefronts per SIMD (128 VGPRs; 3 take 1980 us on the case below): no unit is
// saturated (VALU 35%, LDS 51% busy), the wavefronts wait 60% of their cycles for
// the gathers and for memory-side atomics. 19.8 M items of 64 views on 1.3 M
// faces, all gradients: 2595 us with one thread per face-sorted item, float32 LDS
// sums of the texels and 18 global atomics per run of a face; 1377 us here (TCC
// atomics 44 M -> 13 M). Texture alone, 8.1 M items: 865 -> 328 us.
template <bool LDS_CAMS, bool TEX, bool VTX>
__global__ __launch_bounds__(kBwdThreads, 4) void k_bwd_items(
    const DevView* __restrict__ views, int n_views, DevMesh mesh, const int4* __restrict__ items,
    const int32_t* __restrict__ n_items_p, int rounds, DevGrads g) {
#pragma clang fp contract(fast)
  using Lds = BwdLds<TEX, VTX>;
  __shared__ Lds s;
  const int n_items = *n_items_p;
  const int64_t first = int64_t(blockIdx.x) * kBwdThreads * rounds;
  if (first >= n_items) return;  // whole block idle
  const bool col = VTX && g.colors;  // uniform over the block
  const int tid = threadIdx.x;
  if (TEX)
    for (int j = tid; j < Lds::kTex; j += kBwdThreads) {
      s.tkey[j] = -1;
      s.tval[0][j] = s.tval[1][j] = s.tval[2][j] = 0.0;
    }
  if (VTX)
    for (int j = tid; j < Lds::kVtx; j += kBwdThreads) {
      s.vkey[j] = -1;
      for (int k = 0; k < 6; k++) s.vval[k][j] = 0.0;
    }
  if (LDS_CAMS && tid < n_views) {
    const DevView& v = views[tid];
    BwdCam& c = s.cam[tid];
    c.fx = v.fx;
    c.fy = v.fy;
    c.cx = v.cx;
    c.cy = v.cy;
    for (int k = 0; k < 9; k++) c.R[k] = v.w2c_R[k];
    for (int k = 0; k < 3; k++) c.t[k] = v.w2c_t[k];
    c.grad = v.grad;
  }
  __syncthreads();

  for (int round = 0; round < rounds; round++) {
    const int64_t i = first + int64_t(round) * kBwdThreads + tid;
    const bool valid = i < n_items;
    int4 item = make_int4(-1, 0, 0, 0);
    if (valid) item = items[i];
    const int fid = item.x;
    int vid[3] = {0, 0, 0}, slot[3] = {-1, -1, -1};
    double X[3], Y[3], iZ[3], b1 = 0.0, b2 = 0.0, is = 0.0, gu = 0.0, gv = 0.0;
    const double px = item.z & 0xffff, py = item.z >> 16;
    const CamRef<LDS_CAMS> cam(s.cam, views, item.y);
    float val[9];
    for (int k = 0; k < 9; k++) val[k] = 0.0f;
    if (valid) {
      const int32_t* fi = mesh.faces + int64_t(fid) * 3;
      vid[0] = fi[0];
      vid[1] = fi[1];
      vid[2] = fi[2];
      // everything the item's indices lead to is loaded before any of it is used
      const float* gp = cam.grad() + int64_t(item.w) * 3;
      const float G[3] = {gp[0], gp[1], gp[2]};
      // the corners' uvs: the first 24 bytes of the face's shading record
      const float4* rec = mesh.shade + int64_t(fid) * 4;
      const float4 ab = rec[0];
      const float2 c = *reinterpret_cast<const float2*>(rec + 1);
      float P[9], C[9];
      for (int j = 0; j < 3; j++) {
        const float* q = mesh.verts + int64_t(vid[j]) * 3;
        P[3 * j] = q[0];
        P[3 * j + 1] = q[1];
        P[3 * j + 2] = q[2];
      }
      const float* cols = mesh.vcolors ? mesh.vcolors : mesh.verts;
      for (int j = 0; j < 3; j++) {
        const float* q = cols + int64_t(vid[j]) * 3;
        C[3 * j] = q[0];
        C[3 * j + 1] = q[1];
        C[3 * j + 2] = q[2];
      }
      for (int j = 0; j < 3; j++) {
        const double p0 = P[3 * j], p1 = P[3 * j + 1], p2 = P[3 * j + 2];
        const double qx = cam.R(0) * p0 + cam.R(1) * p1 + cam.R(2) * p2 + cam.t(0);
        const double qy = cam.R(3) * p0 + cam.R(4) * p1 + cam.R(5) * p2 + cam.t(1);
        const double qz = cam.R(6) * p0 + cam.R(7) * p1 + cam.R(8) * p2 + cam.t(2);
        iZ[j] = recip(qz);
        X[j] = cam.fx() * qx * iZ[j] + (cam.cx() - px);
        Y[j] = cam.fy() * qy * iZ[j] + (cam.cy() - py);
      }
      const double q0 = (X[2] * Y[1] - X[1] * Y[2]) * iZ[0];
      const double q1 = (X[0] * Y[2] - X[2] * Y[0]) * iZ[1];
      const double q2 = (X[1] * Y[0] - X[0] * Y[1]) * iZ[2];
      is = recip(q0 + q1 + q2);
      b1 = q1 * is;
      b2 = q2 * is;
      const double b0 = 1.0 - b1 - b2;

      // colour and texture terms: dL/dC, dL/dT and dL/du, dL/dv
      // (dL/dc = G t, dL/dt = G c; u = b1, v = b2, b0 = 1 - u - v)
      float T[12];
      double lu = 0.0, lv = 0.0, dx_du = 0.0, dx_dv = 0.0, dy_du = 0.0, dy_dv = 0.0;
      int cell[4] = {0, 0, 0, 0}, h[4] = {-1, -1, -1, -1};
      if (mesh.ftex) {
        const double iu = b0 * ab.x + b1 * ab.z + b2 * c.x;
        const double iv = b0 * ab.y + b1 * ab.w + b2 * c.y;
        const int tw = mesh.ftex_w, th = mesh.ftex_h;
        const double sx = tw - 1, sy = -(th - 1.0);
        const double fxp = iu * sx, fyp = (1.0 - iv) * (th - 1);
        const double flx = floor(fxp), fly = floor(fyp);
        lu = fxp - flx;
        lv = fyp - fly;
        const int tx0 = clamp_cell(flx, tw - 1), tx1 = clamp_cell(flx + 1.0, tw - 1);
        const int ty0 = clamp_cell(fly, th - 1), ty1 = clamp_cell(fly + 1.0, th - 1);
        dx_du = sx * (double(ab.z) - ab.x);
        dx_dv = sx * (double(c.x) - ab.x);
        dy_du = sy * (double(ab.w) - ab.y);
        dy_dv = sy * (double(c.y) - ab.y);
        for (int q = 0; q < 4; q++) {
          const int x = (q & 1) ? tx1 : tx0, y = (q & 2) ? ty1 : ty0;
          cell[q] = y * tw + x;
          const float* p = mesh.ftex + int64_t(cell[q]) * 3;
          T[3 * q] = p[0];
          T[3 * q + 1] = p[1];
          T[3 * q + 2] = p[2];
          if (TEX)
            h[q] = find_slot<Lds::kTex, Lds::kTex / 4 + 4, kTexProbes>(
                s.tkey, tex_slot<Lds::kTex>(x, y), cell[q]);
        }
      }
      const double ru = 1.0 - lu, rv = 1.0 - lv;
      double glx = 0.0, gly = 0.0;  // dL/d(texel column), dL/d(texel row)
      for (int k = 0; k < 3; k++) {
        const double gk = G[k];
        double t = 1.0, gt = gk;
        if (mesh.ftex) {
          // rows at the column's fraction, then between the rows
          const double d0 = double(T[3 + k]) - T[k], d1 = double(T[9 + k]) - T[6 + k];
          const double r0 = T[k] + lu * d0, r1 = T[6 + k] + lu * d1;
          t = r0 + lv * (r1 - r0);
          if (mesh.vcolors) gt = gk * (b0 * C[k] + b1 * C[3 + k] + b2 * C[6 + k]);
          glx += gt * (d0 + lv * (d1 - d0));
          gly += gt * (r1 - r0);
        }
        if (mesh.vcolors) {
          const double gc = gk * t;
          val[k] = static_cast<float>(gc * b0);
          val[3 + k] = static_cast<float>(gc * b1);
          val[6 + k] = static_cast<float>(gc * b2);
          gu += gc * (double(C[3 + k]) - C[k]);
          gv += gc * (double(C[6 + k]) - C[k]);
        }
        if (TEX) {
          const double g0 = gt * rv, g1 = gt * lv;
          const float v[4] = {static_cast<float>(g0 * ru), static_cast<float>(g0 * lu),
                              static_cast<float>(g1 * ru), static_cast<float>(g1 * lu)};
          for (int q = 0; q < 4; q++) {
            if (h[q] >= 0)
              unsafeAtomicAdd(&s.tval[k][h[q]], double(v[q]));
            else
              unsafeAtomicAdd(&g.texture[int64_t(cell[q]) * 3 + k], v[q]);
          }
        }
      }
      gu += glx * dx_du + gly * dy_du;
      gv += glx * dx_dv + gly * dy_dv;
    }
    if (!VTX) continue;

    // Few runs of equal faces in the wavefront (large faces): their sums by
    // scans, added by each run's last lane, instead of many adds to one
    // address. With many runs every lane adds its own values.
    const int lane = __lane_id();
    const int prev_fid = wave_prev(fid, INT_MIN), next_fid = wave_next(fid, INT_MIN);
    const bool head = valid && (lane == 0 || prev_fid != fid);
    const uint64_t heads = __ballot(head);
    const bool reduce = __popcll(heads) * 4 <= __popcll(__ballot(valid));
    const bool tail = lane == 63 || next_fid != fid;
    const int run = valid ? __popcll(heads & ((2ull << lane) - 1ull)) : -1 - lane;
    const bool add = valid && (!reduce || tail);
    if (add)
      for (int j = 0; j < 3; j++)
        slot[j] = find_slot<Lds::kVtx, 1, kVtxProbes>(
            s.vkey, static_cast<int>(__umulhi(static_cast<uint32_t>(vid[j]) * 2654435761u, Lds::kVtx)),
            vid[j]);
    if (col) {
      if (reduce)
        for (int k = 0; k < 9; k++) val[k] = run_sum(val[k], run);
      if (add) add_corners(s.vval + 3, slot, vid, val, g.colors);
    }
    if (g.verts) {
      for (int k = 0; k < 9; k++) val[k] = 0.0f;
      if (valid) {
        const double S = gu * b1 + gv * b2;
        const double g0 = -S * iZ[0], g1 = (gu - S) * iZ[1], g2 = (gv - S) * iZ[2];
        const double e0 = g0 * is, e1 = g1 * is, e2 = g2 * is;
        const double gX[3] = {e1 * Y[2] - e2 * Y[1], e2 * Y[0] - e0 * Y[2],
                              e0 * Y[1] - e1 * Y[0]};
        const double gY[3] = {e2 * X[1] - e1 * X[2], e0 * X[2] - e2 * X[0],
                              e1 * X[0] - e0 * X[1]};
        const double gZ[3] = {-g0 * (1.0 - b1 - b2), -g1 * b1, -g2 * b2};
        // X + px = fx Qx / Qz + cx, Y + py = fy Qy / Qz + cy, Z = Qz; Q = R P + t
        const double ax = px - cam.cx(), ay = py - cam.cy();
        for (int j = 0; j < 3; j++) {
          const double qx = gX[j] * cam.fx() * iZ[j];
          const double qy = gY[j] * cam.fy() * iZ[j];
          const double qz = gZ[j] - (gX[j] * (X[j] + ax) + gY[j] * (Y[j] + ay)) * iZ[j];
          for (int d = 0; d < 3; d++)
            val[3 * j + d] = static_cast<float>(cam.R(d) * qx + cam.R(3 + d) * qy + cam.R(6 + d) * qz);
        }
      }
      if (reduce)
        for (int k = 0; k < 9; k++) val[k] = run_sum(val[k], run);
      if (add) add_corners(s.vval, slot, vid, val, g.verts);
    }
  }
  __syncthreads();
  // three consecutive lanes write a texel's or vertex's components: one atomic
  // request per 64-byte line they share
  if (TEX)
    for (int j = tid; j < 3 * Lds::kTex; j += kBwdThreads) {
      const int h = j / 3, k = j - 3 * h, key = s.tkey[h];
      if (key >= 0)
        unsafeAtomicAdd(&g.texture[int64_t(key) * 3 + k], static_cast<float>(s.tval[k][h]));
    }
  if (VTX)
    for (int j = tid; j < 3 * Lds::kVtx; j += kBwdThreads) {
      const int h = j / 3, k = j - 3 * h, key = s.vkey[h];
      if (key < 0) continue;
      if (g.verts)
        unsafeAtomicAdd(&g.verts[int64_t(key) * 3 + k], static_cast<float>(s.vval[k][h]));
      if (col)
        unsafeAtomicAdd(&g.colors[int64_t(key) * 3 + k], static_cast<float>(s.vval[3 + k][h]));
    }
}

// Scratch of the backward pass: counts (zero between calls) and cursors.
int64_t backward_scratch_ints() { return 2 * kBwdGroups + 1; }

// Where the item total stands in the scratch after a pass.
int64_t backward_total_at(int32_t F) {
  return kBwdGroups + ((F - 1) >> backward_group_shift(F)) + 1;
}

template <bool TEX, bool VTX>
static void launch_items(hipStream_t st, dim3 grid, const DevView* views, int n_views,
                         const DevMesh& mesh, const int4* items, const int32_t* total, int rounds,
                         const DevGrads& g) {
  if (n_views <= kBwdCams)
    hipLaunchKernelGGL((k_bwd_items<true, TEX, VTX>), grid, dim3(kBwdThreads), 0, st, views, n_views,
                       mesh, items, total, rounds, g);
  else
    hipLaunchKernelGGL((k_bwd_items<false, TEX, VTX>), grid, dim3(kBwdThreads), 0, st, views, n_views,
                       mesh, items, total, rounds, g);
}

// max_squares: 16 x 16 pixel squares of the largest view
int launch_backward(hipStream_t st, const DevView* views, int n_views, int max_squares,
                    int64_t total_pixels, const DevMesh& mesh, const DevGrads& g, int4* items,
                    int32_t* scratch, hipEvent_t before_items) {
  if (max_squares <= 0 || total_pixels <= 0 || mesh.F <= 0) return 0;
  const int F = mesh.F, shift = backward_group_shift(F), groups = ((F - 1) >> shift) + 1;
  int32_t* cnt = scratch;
  int32_t* cursor = scratch + kBwdGroups;
  const dim3 pgrid((max_squares + kBwdSquares - 1) / kBwdSquares, n_views);
  hipLaunchKernelGGL(k_bwd_count, pgrid, dim3(256), 0, st, views, F, shift, cnt);
  hipLaunchKernelGGL(k_bwd_offsets, dim3((groups + 1023) / 1024), dim3(1024), 0, st, cnt, groups,
                     cursor);
  hipLaunchKernelGGL(k_bwd_scatter, pgrid, dim3(256), 0, st, views, F, shift, cnt, cursor, items);
  if (before_items) (void)hipEventRecord(before_items, st);
  // items per thread: few enough that a block's texels fit its table (64 views of
  // 1.3 M faces: 3 per thread 1383 us, 2: 1400, 4: 1420, 8: 2060), fewer where the
  // blocks would not fill the chip; at most one item per pixel, blocks past the
  // item total exit at once
  const int rounds = total_pixels >= (int64_t(1) << 22) ? 3 : total_pixels >= (int64_t(1) << 20) ? 2 : 1;
  const int64_t per = int64_t(kBwdThreads) * rounds;
  const dim3 grid(static_cast<unsigned>((total_pixels + per - 1) / per));
  const bool tex = g.texture && mesh.ftex, vtx = g.verts || (g.colors && mesh.vcolors);
  const int32_t* total = cursor + groups;
  if (tex && vtx)
    launch_items<true, true>(st, grid, views, n_views, mesh, items, total, rounds, g);
  else if (tex)
    launch_items<true, false>(st, grid, views, n_views, mesh, items, total, rounds, g);
  else if (vtx)
    launch_items<false, true>(st, grid, views, n_views, mesh, items, total, rounds, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace ugu_hip
