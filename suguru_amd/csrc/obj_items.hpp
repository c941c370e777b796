// obj_items.hpp -- how the spread by capsule objects cuts an object's box into work items, and how
// many items its buffers hold (constant expressions: the same on host and device).
#pragma once

namespace ibx {

constexpr int OB_BX = 32;    // item extent limit in x and y (cells)
constexpr int OB_NZ = 32;    // item extent limit in z
constexpr int OB_NC = 2048;  // cells per item

// Extent of the items of a launch: at most bx cells in x and y and nc cells.
struct ObjLimit {
  int bx, nc;
};

// The extents that a launch chooses from: 2048, 1024, 512 and 256 cells.
constexpr int OB_LIMITS = 4;
constexpr ObjLimit obj_limit(int e) { return {e ? OB_BX / 2 : OB_BX, OB_NC >> e}; }

// Item grid of one object box (its bounds xa, xb, ya, yb, za, zb): cx x cy x cz sub-boxes of extent
// nx x ny x nz (the last ones cut short), within the launch's limit and OB_NZ planes each.
struct ObjGrid {
  int cx, cy, cz, nx, ny, nz;
  constexpr ObjGrid(const int* b, ObjLimit l)
      : ObjGrid(b[1] - b[0] + 1, b[3] - b[2] + 1, b[5] - b[4] + 1, l) {}
  constexpr ObjGrid(int X, int Y, int Z, ObjLimit l) : cx(0), cy(0), cz(0), nx(0), ny(0), nz(0) {
    cx = (X + l.bx - 1) / l.bx, cy = (Y + l.bx - 1) / l.bx;
    nx = (X + cx - 1) / cx, ny = (Y + cy - 1) / cy;
    const int most = Z < OB_NZ ? Z : OB_NZ, fit = l.nc / (nx * ny);
    nz = most < fit ? most : fit;
    if (nz < 1) nz = 1;
    cz = (Z + nz - 1) / nz;
  }
  constexpr int count() const { return cx * cy * cz; }
};

// Items that the buffers hold for ncap capsules.  By the capsule count alone and never fewer for
// more capsules: a call with fewer capsules than an earlier one leaves the buffers where they are,
// which a captured graph of the earlier call relies on.
constexpr long long obj_item_capacity(long long ncap) {
  return 64 * (ncap < 16 ? 16 : ncap) + 1024;
}

// The limit of a launch whose boxes make tot[e] items at each: 2048 cells where there are enough of
// them to fill the chip, fewer where a capsule or a few would otherwise leave it idle: an item is one
// workgroup's chain over its candidates, so that smaller items end sooner, while candidates near an
// item's faces are prepared once for each item they reach.  The lines lie at the items of 2048
// cells, counted from the boxes.  Capsules of degree 16 and radius 10.6h (8 items each) on
// 256 x 256 x 128 cells, spread with items of 2048 / 1024 / 512 / 256 cells: 1 (8 items) 93 / 78 / 76 /
// 75 us; 8 (64) 98 / 86 / 80 / 82; 16 (127) 106 / 91 / 87 / 101; 24 (190) 107 / 99 / 91 / 121;
// 30 (240) 105 / 96 / 93 / 131; 45 (360) 108 / 96 / 109 / 155; 60 (480) 107 / 108 / 120 / 180;
// 76 (600) 116 / 119 / 138 / 221; 100 (790) 122 / 134 / 158 / 255; 226 (1790) 203 / 226 / 284 / 534.
// Spread and interpolation on a denser channel: 4 (32) 156 / 132 / 117 / 105; 16 162 / 130 / 118 / 129;
// 30 171 / 138 / 144 / -; 60 181 / 160 / 177 / -; 1000 1108 / 1306 / 1725 / -.
// Smaller items are taken only where the buffers hold them: the next larger ones otherwise.  (The
// largest are taken whether they fit or not, and their overflow reported.)
constexpr int obj_choice(const int* tot, int icap) {
  int e = tot[0] <= 48 ? 3 : tot[0] <= 200 ? 2 : tot[0] <= 500 ? 1 : 0;
  for (int l = OB_LIMITS - 1; l > 0; --l)  // (constant indices: tot may be registers)
    if (e == l && tot[l] > icap) e = l - 1;
  return e;
}

// Counts of the three smaller limits in one word, 21 bits each, saturated.
constexpr int OB_CBITS = 21, OB_CMAX = 1 << 20;
constexpr unsigned long long obj_pack(const int* cnt) {
  unsigned long long v = 0;
  for (int e = 1; e < OB_LIMITS; ++e)
    v |= (unsigned long long)(cnt[e] < OB_CMAX ? cnt[e] : OB_CMAX) << (OB_CBITS * (e - 1));
  return v;
}
constexpr int obj_unpack(unsigned long long v, int e) {
  return (int)(v >> (OB_CBITS * (e - 1))) & ((1 << OB_CBITS) - 1);
}

}  // namespace ibx
