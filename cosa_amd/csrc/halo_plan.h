// halo_plan.h -- host checks of a level's BC patches and cuts, free of HIP so
// that they can be tested alone.  Blocks have imax, jmax, kmax (nodes); patches
// block, type, t (bctopo); cuts b1, b2, t (cutopo).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdlib>
#include <vector>

namespace cosahip {

// Host replica of k_cut's index arithmetic: every halo target and interior
// source of the cut must lie inside its block's P3 extents.
template <class Block>
bool cut_in_bounds(const Block& b1, const Block& b2, const int* t, int n2, int count) {
  const int idir1 = t[1], inout1 = t[2], idir2 = t[10], inout2 = t[11];
  int istr1[4], iend1[4], istr2[4], iend2[4], iord[4];
  istr1[1] = t[3]; iend1[1] = t[4]; istr1[2] = t[5]; iend1[2] = t[6]; istr1[3] = t[7]; iend1[3] = t[8];
  istr2[1] = t[12]; iend2[1] = t[13]; istr2[2] = t[14]; iend2[2] = t[15]; istr2[3] = t[16]; iend2[3] = t[17];
  iord[1] = t[18]; iord[2] = t[19]; iord[3] = t[20];
  for (int m = 1; m <= 3; m++)
    if (iord[m] < 1 || iord[m] > 3) return false;
  const int ijk1[4] = {0, b1.imax, b1.jmax, b1.kmax}, ijk2[4] = {0, b2.imax, b2.jmax, b2.kmax};
  const int ibcpt = inout1 == 1 ? 0 : ijk1[idir1], ibcinc = inout1 == 1 ? -1 : 1;
  const int inr = inout2 == 1 ? 1 : ijk2[idir2] - 1, inrinc = inout2 == 1 ? 1 : -1;
  auto cyc = [](int d, int m) { return (d - 1 + m - 1) % 3 + 1; };
  const int ic1 = cyc(idir1, 1), ic2 = cyc(idir1, 2), ic3 = cyc(idir1, 3);
  const int jc1 = iord[ic1], jc2 = iord[ic2], jc3 = iord[ic3];
  const int sg1c2 = iend1[ic2] > istr1[ic2] ? 1 : -1, sg1c3 = iend1[ic3] > istr1[ic3] ? 1 : -1;
  const int sg2c2 = iend2[jc2] > istr2[jc2] ? 1 : -1, sg2c3 = iend2[jc3] > istr2[jc3] ? 1 : -1;
  auto inside = [](const Block& b, int i, int j, int k) {
    return i >= -1 && i <= b.imax + 1 && j >= -1 && j <= b.jmax + 1 && k >= -1 && k <= b.kmax + 1;
  };
  for (int item = 0; item < count; item++) {
    const int i2_ = item % n2, i3_ = item / n2;
    const int a2 = istr1[ic2] + sg1c2 * i2_, a3 = istr1[ic3] + sg1c3 * i3_;
    int x1[4] = {0, 0, 0, 0};
    x1[ic1] = ibcpt;
    x1[ic2] = a2;
    x1[ic3] = a3;
    int x2[4] = {0, x1[1], x1[2], x1[3]};
    x2[ic1] += ibcinc;
    const int c2 = istr2[jc2] + sg2c2 * i2_, c3 = istr2[jc3] + sg2c3 * i3_;
    int y1[4] = {0, 0, 0, 0};
    y1[jc1] += inr;   // sums, as in bc_ijk, where the order repeats an axis
    y1[jc2] += c2;
    y1[jc3] += c3;
    int y2[4] = {0, y1[1], y1[2], y1[3]};
    y2[jc1] += inrinc;
    if (!inside(b1, x1[1], x1[2], x1[3]) || !inside(b1, x2[1], x2[2], x2[3]) || !inside(b2, y1[1], y1[2], y1[3]) ||
        !inside(b2, y2[1], y2[2], y2[3]))
      return false;
  }
  return true;
}

// What the halo fill of a level may be relied on for.
// fresh: every face-halo cell of every block is set by each fill, from
// interior cells alone.  A wall, symmetry or cut record reads two cells deep,
// so in a block one cell thick it reads the far halo; a face that no record
// covers keeps what it holds.
// once: besides, each is set by exactly one point of one patch or cut, and
// no block is one cell thick: then the halo fill and bprtest may run as one
// launch (k_halo) -- no order between patches and cuts matters, and the cells
// they set are all the halo cells bprtest looks at.
struct HaloPlan {
  bool fresh, once;
};
template <class Blocks, class Patches, class Cuts>
HaloPlan plan_halos(const Blocks& blks, const Patches& patches, const Cuts& cuts) {
  std::vector<std::vector<unsigned char>> hit(6 * (size_t)blks.size());
  bool fresh = true, once = true;
  auto ext = [&](int b, int d) {
    const auto& B = blks[b];
    return (d == 1 ? B.imax : d == 2 ? B.jmax : B.kmax) - 1;
  };
  auto mark = [&](int block, int idir, int inout, int c2lo, int c2hi, int c3lo, int c3hi) {
    // transverse extents in the cyclic order of the record
    const int e2 = ext(block, idir % 3 + 1), e3 = ext(block, (idir + 1) % 3 + 1);
    auto& h = hit[6 * (size_t)block + 2 * (idir - 1) + (inout == 1 ? 0 : 1)];
    if (h.empty()) h.assign((size_t)e2 * e3, 0);
    if (c2lo < 1 || c3lo < 1 || c2hi > e2 || c3hi > e3) once = false;
    for (int c3 = std::max(c3lo, 1); c3 <= std::min(c3hi, e3); c3++)
      for (int c2 = std::max(c2lo, 1); c2 <= std::min(c2hi, e2); c2++) {
        unsigned char& c = h[(size_t)(c3 - 1) * e2 + c2 - 1];
        if (c) once = false;
        c = 1;
      }
  };
  for (const auto& B : blks)
    if (B.imax < 3 || B.jmax < 3 || B.kmax < 3) once = false;
  for (const auto& r : patches) {
    const int i2 = r.t[1] % 3 + 1, i3 = (r.t[1] + 1) % 3 + 1;
    mark(r.block, r.t[1], r.t[2], r.t[2 * i2 + 1], r.t[2 * i2 + 2], r.t[2 * i3 + 1], r.t[2 * i3 + 2]);
    if (r.type != 30 && r.type != 4 && ext(r.block, r.t[1]) < 2) fresh = false;
  }
  for (const auto& r : cuts) {
    const int i2 = r.t[1] % 3 + 1, i3 = (r.t[1] + 1) % 3 + 1;
    const int a2 = r.t[2 * i2 + 1], b2 = r.t[2 * i2 + 2], a3 = r.t[2 * i3 + 1], b3 = r.t[2 * i3 + 2];
    mark(r.b1, r.t[1], r.t[2], std::min(a2, b2), std::max(a2, b2), std::min(a3, b3), std::max(a3, b3));
    // the sources: interior cells of block 2 (cut_in_bounds allows its halos).
    // The two cells off face 2 lie along the axis that the normal of face 1 is
    // mapped to, so that has to be the normal of face 2, and the order has to
    // be one of all three axes.
    const int* ord = r.t + 17;
    if (ord[r.t[1]] != r.t[10] || ord[1] == ord[2] || ord[1] == ord[3] || ord[2] == ord[3]) fresh = false;
    if (ext(r.b2, r.t[10]) < 2) fresh = false;
    for (int m = 1; m <= 2; m++) {
      const int d = ord[(r.t[1] + m - 1) % 3 + 1], len = m == 1 ? b2 - a2 : b3 - a3;
      const int lo = r.t[10 + 2 * d], sg = r.t[11 + 2 * d] > lo ? 1 : -1;
      const int hi = lo + sg * std::abs(len);
      if (std::min(lo, hi) < 1 || std::max(lo, hi) > ext(r.b2, d)) fresh = false;
    }
  }
  for (const auto& h : hit)
    if (h.empty() || std::find(h.begin(), h.end(), 0) != h.end()) fresh = false;
  return HaloPlan{fresh, fresh && once};
}

}  // namespace cosahip
