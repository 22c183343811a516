// Binning of faces into screen tiles, shared by the rasterizer's and the
// raytracer's tile kernels: wavefront-aggregated appends to the tiles' bins,
// the bin entries' order and the hidden-face test.
#pragma once

#include "device_common.h"

#pragma clang fp contract(off)

namespace ugu_hip {

// Views per thread: the face's indices are loaded once and reused for
// kSetupViews consecutive views (grid.y = ceil(n_views / kSetupViews)).
constexpr int kSetupViews = 8;

// Bin appends a setup thread issues before waiting for their atomics: a face
// whose pixel bbox spans up to this many tiles costs one atomic round trip
// per view.
constexpr int kAppendRounds = 4;

// Faces whose pixel bbox holds at most this many pixel centres are tested at
// those centres before they are binned.
constexpr int kCoverProbe = 4;

// Appends `entry` to a bin segment for every lane with `has`, in two halves.
// `seg` = 4 * tile for the front segment (filled upwards from the bin's first
// slot) and 4 * tile + 1 for the back segment (filled downwards from its last
// slot). append_issue groups the lanes that target the same segment (ballot +
// popcount rank) and the group leaders issue their atomicAdds together;
// append_finish broadcasts each group's base and stores the entries. A caller
// issues several appends before finishing any, so the wavefront waits for
// one atomic round trip for all of them. Entries of one segment are in no
// particular order (the rasterizer's result does not depend on it). When the
// two segments together overflow the bin they overwrite each other's slots;
// every slot the rasterizer reads still holds a valid entry, and the host
// renders again with larger bins.
struct AppendTicket {
  int ret;   // the group's first slot, in the leader lane
  int lr;    // leader lane | rank in the group << 8
  int seg;   // segment, -1 for lanes without an entry
};

// Lower bound of the skip depths of a wavefront's back-face entries (bits of
// a non-negative float; 0 when one has no bound): the leaders of back groups
// fold it into their tile's back-segment minimum.
UGU_DEV uint32_t back_zmin(bool back, float zskip) {
  uint32_t zmin = 0xffffffffu;
  if (__ballot(back))
    zmin = wave_min_u32(back ? (zskip >= 0.0f ? __float_as_uint(zskip) : 0u) : 0xffffffffu);
  return zmin;
}

UGU_DEV AppendTicket append_issue(const DevBins& bins, int seg, uint32_t zmin, bool has) {
  AppendTicket tk;
  tk.ret = 0;
  tk.lr = 0;
  tk.seg = has ? seg : -1;
  const uint64_t hasm = __builtin_amdgcn_ballot_w64(has);
  if (!hasm) return tk;
  // Each pass takes the lowest pending lane; the lanes with its segment form
  // one group, whose lowest lane (that one) leads it. A lane keeps its
  // group's mask; rank, leader and size follow from it after the loop.
  uint64_t todo = hasm, grp_mine = 0;
  while (todo) {
    const int l = __ffsll(static_cast<unsigned long long>(todo)) - 1;
    const int ls = __builtin_amdgcn_readlane(seg, l);
    const uint64_t grp = __builtin_amdgcn_ballot_w64(seg == ls) & hasm;
    grp_mine = (has && seg == ls) ? grp : grp_mine;
    todo &= ~grp;
  }
  const int rank = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
      static_cast<uint32_t>(grp_mine >> 32),
      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(grp_mine), 0u)));
  if (has && rank == 0) {
    tk.ret = atomicAdd(&bins.counts[seg], __popcll(grp_mine));
    if (seg & 1) atomicMin(reinterpret_cast<unsigned int*>(bins.counts) + (seg + 1), zmin);
  }
  const int leader = has ? __ffsll(static_cast<unsigned long long>(grp_mine)) - 1 : 0;
  tk.lr = leader | (rank << 8);
  return tk;
}

// Finishes the first `used` (wavefront-uniform) of R tickets: every group
// base is broadcast before the first store, so the wavefront waits once for
// all its atomics (a store issued before a later wait would be waited for as
// well).
// With PER_ROUND every round has an entry of its own, and a lane whose slot
// lies past its bin's end publishes the occupancy it saw (status[0]).
template <int R, bool PER_ROUND = false>
UGU_DEV void append_finish(const DevBins& bins, const AppendTicket* tk, const int2* entry,
                           int used = R) {
  int slot[R];
#pragma unroll
  for (int r = 0; r < R; r++)
    slot[r] = r < used ? __shfl(tk[r].ret, tk[r].lr & 0xff) + (tk[r].lr >> 8) : 0;
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (r < used && tk[r].seg >= 0) {
      if (slot[r] < bins.cap) {
        const int64_t row = int64_t(tk[r].seg >> 2) * bins.cap;
        bins.bins[row + ((tk[r].seg & 1) ? bins.cap - 1 - slot[r] : slot[r])] =
            PER_ROUND ? entry[r] : *entry;
      } else if (PER_ROUND) {
        atomicMax(&bins.status[0], slot[r] + 1);
      }
    }
  }
}

// Entry i of a tile's bin: the front segment's nA entries, then the back
// segment read from the bin's last slot downwards.
// Each entry is read once, so the load is non-temporal: the stream of entries
// does not evict the face records, shading records and texels the rasterizer
// reads again (64-view batch: rasterizer -2%).
UGU_DEV int2 bin_entry(const int2* bin, int nA, int cap, int i) {
  const int2* p = i < nA ? bin + i : bin + (cap - 1 - (i - nA));
  const long long q = __builtin_nontemporal_load(reinterpret_cast<const long long*>(p));
  return make_int2(static_cast<int>(q & 0xffffffffll), static_cast<int>(q >> 32));
}

// True when the tile's current depth bound proves the face hidden.
UGU_DEV bool skip_face(float zskip, float dmax) {
  return dmax >= 1e-18f && zskip > dmax * 1.00390625f;
}

// (face, pixel) pairs of a tile's chunk of NT staged faces (NT threads, one face
// slot each), numbered slot by slot.
template <int NT>
struct PairLds {
  uint16_t pre[NT];          // pairs before the slot's among its wavefront's slots
  int32_t wsum[2][NT / 64];  // pairs of each wavefront's slots, by chunk parity
  int32_t mark[NT];          // starts of the faces of a wavefront's 64 pairs
  uint16_t queue[2 * NT];    // a wavefront's pairs that passed the first test
};

// Publishes this thread's pair count; a barrier and walk_pairs follow. The
// parity of the chunk keeps a wavefront that has gone on to the next chunk from
// overwriting the sums that a slower one still reads.
template <int NT>
UGU_DEV void publish_pairs(PairLds<NT>& s, int parity, int c) {
  const int x = wave_incl_sum(c);
  s.pre[threadIdx.x] = static_cast<uint16_t>(x - c);  // at most 64 NT - 1
  if ((threadIdx.x & 63) == 63) s.wsum[parity][threadIdx.x >> 6] = x;
}

// Runs first(slot, r, pix) for every pair (r: the pair's index in its face,
// 0 <= r < NT; it sets the tile pixel) and second(slot, pix) for those where first
// returned true, 64 of them at a time (ALL: where it returns true for all of
// them). Returns the number of pairs.
// Each wavefront takes 64 consecutive pairs at a time without the others: every
// lane holds the first pairs of NT / 64 slots, marks those in the wavefront's
// window at their place in LDS, and a running maximum carries each mark to the
// pairs of its face. The cost does not depend on the faces' sizes (a list that
// each face's thread writes costs the largest face's pairs, a binary search per
// pair eight dependent LDS reads), and no barrier lies between two windows.
template <int NT, bool ALL = false, class First, class Second>
UGU_DEV int walk_pairs(PairLds<NT>& s, int parity, First first, Second second) {
  constexpr int K = NT / 64;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int base = 0, total = 0;
#pragma unroll
  for (int w = 0; w < K; w++) {
    if (w < lane * K / 64) base += s.wsum[parity][w];
    total += s.wsum[parity][w];
  }
  if (total == 0) return 0;
  int q[K + 1];
#pragma unroll
  for (int k = 0; k < K; k++) q[k] = base + s.pre[lane * K + k];
  q[K] = __shfl_down(q[0], 1);
  if (lane == 63) q[K] = total;
  int32_t* mark = s.mark + wid * 64;
  uint16_t* queue = s.queue + wid * 128;
  int queued = 0;
  for (int g = wid * 64; g < total; g += NT) {
    // mark = slot << 17 | (first pair - g + 65536); a face that starts before the
    // window marks its first place
    mark[lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int k = 0; k < K; k++)
      if (q[k] < q[k + 1] && q[k + 1] > g && q[k] < g + 64)
        mark[max(q[k] - g, 0)] = ((lane * K + k) << 17) | (q[k] - g + 65536);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int m = wave_incl_max(mark[lane]);
    const int j = m >> 17;
    int pix = 0;
    const bool keep = g + lane < total && first(j, lane + 65536 - (m & 0x1ffff), pix);
    if (ALL) {
      if (keep) second(j, pix);
      continue;
    }
    const uint64_t kept = __builtin_amdgcn_ballot_w64(keep);
    if (keep)
      queue[queued + static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                         static_cast<uint32_t>(kept >> 32),
                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(kept), 0u)))] =
          static_cast<uint16_t>(j | (pix << 8));
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    queued += __popcll(kept);
    if (queued >= 64) {
      queued -= 64;
      const int e = queue[queued + lane];
      second(e & 0xff, e >> 8);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (lane < queued) {
    const int e = queue[lane];
    second(e & 0xff, e >> 8);
  }
  return total;
}

// Row of pair r in a box nx pixels wide (r, nx < 1024): r / nx, as the quotient
// of r + 1/2 is at least 1 / (2 nx) away from an integer.
UGU_DEV int pair_row(int r, int nx) {
  return static_cast<int>((static_cast<float>(r) + 0.5f) *
                          __builtin_amdgcn_rcpf(static_cast<float>(nx)));
}

}  // namespace ugu_hip
