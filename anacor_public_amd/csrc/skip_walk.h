// The skip walk: the tracer's A_h kernel on a field of free distances.
// Included by trace.hip inside namespace anacor, after the stepping kernels.
//
// The reference visits every voxel of a ray, although all that a ray's result
// depends on is how many of its steps fall on each label, where it stops and
// its last voxel.  Crystal, loop and liquor are regions tens of voxels thick,
// so nearly all steps repeat the label of the step before.  Per voxel and
// direction octant the field holds one byte: the label (bits 0-2) and 8 n (bits
// 3-7), where n is the side (in voxels, at most 31) of a cube that starts at the
// voxel, extends into the octant and holds that one label.  A ray of the octant
// whose steps move at most one voxel per axis stays in that cube for n - 1 more
// steps, so one gather answers n steps: 13 gathers per ray in place of 101 steps on a
// 256^3 volume (18 against 117 in a wave's longest lane), with the same step
// counts per label.
//
// Positions are exact without FP64 in the loop.  The reference evaluates
// rnd(c + RN(inc * d)) per stepped axis, c an integer; that is c + rnd(m),
// m = RN(inc * d), unless c + m rounds up onto the boundary of rnd, which
// takes an m within 2^-40 below a boundary.  So the offsets from a ray's
// origin depend on (ray, exit face, increment) only: each workgroup tabulates
// them in LDS for its reflection and notes the first increment of each face
// that is too close to call.  A lane that would use it, or whose geometry the
// table does not cover in any other way, marks its reflection (kRayRedo), and
// the host traces such reflections with the stepping kernels.  Where the
// reference aborts, the walk raises the same error itself.
//
// Layout of one octant's field: the volume with a one-voxel replicated shell
// (the reference clamps a stepped coordinate to the volume), tiles of 8 (x) by
// 16 (y) bytes, one 128-byte line each, so the 64 rays of a wave (neighbours
// in Morton order) touch about 15 lines per gather against 29 in rows.  x's
// high bits follow the tile's 7 bits, y's high bits and then z above them: an
// offset adds to a position in two words, x and yz, whose gaps the table's
// words fill with ones so that carries run through, and one bit select merges
// them.
//
// What bounds it: VALU issue (75% of one instruction per SIMD every 4 cycles)
// and the texture addresser (81% busy, 20 cycles per 64-lane byte gather), at
// once.  256^3, 25,323 voxels, 20,000 reflections: 62.5 ms stepping, 21.6 ms
// with the first form of this kernel (507 VALU instructions per wave and ray,
// five waves per SIMD), 17.7 ms with nine instructions per gather and eight
// waves, 13.8 ms with the diffracted ray leading the sort and rows of lanes
// within cubes, 13.4 ms with the errors in LDS.  181x203x227, 5,003 voxels, 4,001
// reflections, FP64 mean: 5.1 and 0.95 ms.

constexpr unsigned kRayRedo = 1u << 30;   // err bit: trace with the stepping kernels
constexpr int kSkipMaxExtent = 2046;      // coordinates in 16 bits, tables in LDS
constexpr int kSkipVox = 4;               // voxels per lane between two table builds
constexpr unsigned kSkipTableBytes = 50000;   // of the tables, beside 14 KB in 64 KB of LDS
constexpr int kLevels = 12;
// cubes of k + 1 voxels: n - 1 is quantised down to these
constexpr int kLevelSide[kLevels] = {1, 2, 3, 4, 5, 6, 7, 8, 12, 16, 24, 30};

struct FieldShape {
  int Z, Y, X;          // volume
  int nbx, nby;         // tiles of 8 and 16 along padded x and y
  int hx;               // bits of the x tile index
  int zs;               // bytes per z plane
  long long bytes;      // per octant
  int wx;               // 32-bit words per padded row of a level plane
};

__host__ __device__ __forceinline__ unsigned dilate_x(int x) {
  return (unsigned)((x & 7) + (x >> 3) * 128);
}
__host__ __device__ __forceinline__ unsigned dilate_y(int y, int hx) {
  return (unsigned)(((y & 15) << 3) + (y >> 4) * (1 << (7 + hx)));
}

// -------------------------------------------------------- building the field
//
// Level k of the bit planes: the cube [p, p + k]^3 (its part inside the padded
// volume) holds one label.  Level 1 compares labels; a level a + s, s <= a, is
// the AND of level a at the eight offsets {0, s}^3 (cubes that share voxels, so
// their labels agree), 32 voxels per word operation.  The cube of octant o at v starts at v - k on o's negative axes,
// so one set of planes serves all eight octants.

__device__ __forceinline__ int padded_label(const uint8_t* __restrict__ vol, int Z, int Y, int X,
                                            int z, int y, int x) {
  const int cz = min(max(z, 1), Z), cy = min(max(y, 1), Y), cx = min(max(x, 1), X);
  return vol[((size_t)cz * (Y + 2) + cy) * (X + 2) + cx];   // the raw layout's zero shell
}

// flag |= 4 when some listed voxel's label is not 3.
__global__ void origin_label_kernel(const uint8_t* __restrict__ vol, int Y, int X,
                                    const int4* __restrict__ coords, int n,
                                    unsigned* __restrict__ flag) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  bool other = false;
  if (i < n) {
    const int4 c = coords[i];
    other = vol[((size_t)(c.x + 1) * (Y + 2) + c.y + 1) * (X + 2) + c.z + 1] != 3;
  }
  if (__any(other) && (threadIdx.x & (kWave - 1)) == 0) atomicOr(flag, 4u);
}

// Level 1: one wave per 64 voxels of a padded row; bits past the row are 1.
__global__ void field_base_kernel(const uint8_t* __restrict__ vol, int Z, int Y, int X, int wx,
                                  long long waves, uint32_t* __restrict__ out) {
  const long long w = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  if (w >= waves) return;               // whole waves
  const int lane = (int)threadIdx.x & (kWave - 1);
  const int per_row = (wx + 1) / 2;
  const long long row = w / per_row;
  const int x = (int)(w - row * per_row) * kWave + lane;
  const int z = (int)(row / (Y + 2)), y = (int)(row - (long long)z * (Y + 2));
  // the label of the 2 x 2 column (z, z + 1) x (y, y + 1) at x, or 255
  auto column = [&](int cx) {
    const int a = padded_label(vol, Z, Y, X, z, y, cx);
    const bool same = padded_label(vol, Z, Y, X, z, y + 1, cx) == a &&
                      padded_label(vol, Z, Y, X, z + 1, y, cx) == a &&
                      padded_label(vol, Z, Y, X, z + 1, y + 1, cx) == a;
    return same ? a : 255;
  };
  const int c0 = column(x);
  int c1 = __shfl_down(c0, 1);
  if (lane == kWave - 1) c1 = column(x + 1);
  const unsigned long long b = __ballot(x >= X + 2 || (c0 != 255 && c1 == c0));
  const int word = (x - lane) / 32 + lane;
  if (lane < 2 && word < wx) out[row * wx + word] = (uint32_t)(b >> (32 * lane));
}

struct ErodeArgs {
  const uint32_t* in;
  uint32_t* out[4];
  int s[4];
  int n;
  int Z2, Y2, wx;       // padded extents, words per row
};

// Up to four levels from one: AND over the offsets {0, s}^3, 1 outside.
__global__ void field_erode_kernel(ErodeArgs a) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)a.Z2 * a.Y2 * a.wx) return;
  const int w = (int)(i % a.wx);
  const long long row = i / a.wx;
  const int y = (int)(row % a.Y2), z = (int)(row / a.Y2);
  for (int k = 0; k < a.n; ++k) {
    const int s = a.s[k];
    uint32_t v = ~0u;
    for (int dz = 0; dz < 2; ++dz)
      for (int dy = 0; dy < 2; ++dy) {
        if (z + dz * s >= a.Z2 || y + dy * s >= a.Y2) continue;
        const uint32_t* p = a.in + ((long long)(z + dz * s) * a.Y2 + (y + dy * s)) * a.wx + w;
        const uint32_t lo = p[0], hi = w + 1 < a.wx ? p[1] : ~0u;
        v &= lo & ((lo >> s) | (hi << (32 - s)));     // 1 <= s <= 16
      }
    a.out[k][i] = v;
  }
}

// Eight x neighbours of one padded (z, y) per thread, all eight octants:
// n from the highest level whose cube holds, clamped to the padded volume on
// the negative side (a cube cut off there is only smaller); 1 for label 0.  What
// bounds it: the latency of the planes' words.  256^3 355 us octant by octant,
// 193 us so; 400x420x450 1,689 and 870 us.
__global__ void field_pack_kernel(const uint8_t* __restrict__ vol, FieldShape s,
                                  const uint32_t* __restrict__ planes, long long plane_words,
                                  uint8_t* __restrict__ field) {
  const int Z2 = s.Z + 2, Y2 = s.Y + 2;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)Z2 * s.nby * s.nbx * 16) return;
  const int yl = (int)(i & 15);
  const long long t = i >> 4;
  const int xb = (int)(t % s.nbx);
  const long long u = t / s.nbx;
  const int yb = (int)(u % s.nby), z = (int)(u / s.nby);
  const int y = yb * 16 + yl, x0 = xb * 8;
  if (y >= Y2) return;
  uint32_t lab[2] = {0x08080808u, 0x08080808u}, keep[2] = {0, 0};   // n = 1; where more counts
  for (int e = 0; e < 8; ++e) {
    const uint32_t l = (uint32_t)padded_label(vol, s.Z, s.Y, s.X, z, y, x0 + e) & 7u;
    lab[e >> 2] |= l << (8 * (e & 3));
    keep[e >> 2] |= (l ? 0xf8u : 0u) << (8 * (e & 3));
  }
  const long long at = (long long)z * s.zs + (long long)yb * (1ll << (7 + s.hx)) +
                       ((long long)xb << 7) + (yl << 3);
  // every octant at once, level by level (their loads are independent), until the
  // cubes of all eight hold nowhere; none count where all labels are 0
  uint32_t acc[8][2] = {};
  unsigned live = (keep[0] | keep[1]) ? 0xffu : 0u;
  int prev = 0;
  for (int l = 0; live && l < kLevels; ++l) {
    const int k = kLevelSide[l];
    const uint32_t add = (uint32_t)(k - prev) << 3;
    prev = k;
    const uint32_t* const plane = planes + l * plane_words;
#pragma unroll
    for (int o = 0; o < 8; ++o) {        // bit 2: z falls, bit 1: y falls, bit 0: x falls
      const int qz = (o & 4) ? max(z - k, 0) : z;
      const int qy = (o & 2) ? max(y - k, 0) : y;
      const uint32_t* row = plane + ((long long)qz * Y2 + qy) * s.wx;
      const int xs = (o & 1) ? x0 - k : x0;
      const int b0 = max(xs, 0), w = b0 >> 5;
      const uint32_t hi = w + 1 < s.wx ? row[w + 1] : ~0u;
      uint32_t bits = (uint32_t)((((uint64_t)hi << 32) | row[w]) >> (b0 & 31));
      if (o & 1) {                       // positions below 0 take row position 0
        const int n = min(max(-xs, 0), 8);
        bits = (bits << n) | ((bits & 1u) ? (1u << n) - 1u : 0u);
      }
      bits &= (live >> o & 1u) ? 0xffu : 0u;
      live &= bits ? ~0u : ~(1u << o);   // higher levels hold larger cubes
      acc[o][0] += (((bits & 15u) * 0x00204081u) & 0x01010101u) * add;
      acc[o][1] += (((bits >> 4) * 0x00204081u) & 0x01010101u) * add;
    }
  }
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    uint2 v;
    v.x = (acc[o][0] & keep[0]) + lab[0];
    v.y = (acc[o][1] & keep[1]) + lab[1];
    *(uint2*)(field + (long long)o * s.bytes + at) = v;
  }
}

// ------------------------------------------------------------- the kernel

struct SkipArgs {
  const uint8_t* field;        // eight octants
  long long oct_bytes;
  int hx, zs;                  // zs: bytes per z plane; in cells, tiles per z plane
  const uint8_t* fine;         // cells: labels of single voxels,
  unsigned fine_bytes;
  int fine_shift;              // 2^fine_shift to a byte
  const int4* vox;             // (z | y << 16, x, x word, yz word), wave-grouped
  const int* index;            // the caller's index of each of them
  int lo[3], hi[3];            // the listed voxels' box (z, y, x): bounds the tables
  int at[3];                   // first table entry of each exit axis
};

// The exit along one axis: the upper plane where the direction's sign bit is
// clear, else the lower one.  Uniform in a workgroup.
struct AxisExit {
  bool up, round;
  int face;                    // index of the face (0..5)
  int add;                     // increments tried past the distance to the plane
  __device__ __forceinline__ AxisExit(const RayRule* __restrict__ rr, int axis) {
    const unsigned hi =
        (unsigned)((unsigned long long)__double_as_longlong(rr->dir[axis]) >> 32);
    up = __builtin_amdgcn_readfirstlane((int)((hi >> 31) ^ rr->neg)) == 0;
    face = axis == 0 ? (up ? 2 : 1) : axis == 1 ? (up ? 4 : 3) : (up ? 0 : 5);
    const uint32_t meta = rr->meta[face];
    round = (meta & kMetaRound) != 0;
    add = up ? ((meta & kMetaInclusive) ? 1 : 0) : 1;
  }
};

// What a lane needs of its exit axis, read from LDS by the axis.
struct AxisLds {
  int at;                      // byte offset of its table
  int near;                    // increments from here on are not tabulated (0: none;
                               // -1: the reference aborts on rays leaving here)
  int scale, add;
  int hb, hc;                  // extents - 1 of the two stepped axes
  int face, up;
  double db, dc;               // deltas of the two stepped axes
  double vb, vc, vp, bias;     // voxel edges: stepped axes, exit axis; rounding bias
};
static_assert(sizeof(AxisLds) == 80, "AxisLds layout");

// Whether the walk may leave along `axis`: the face's precondition holds, and
// its deltas agree with the direction that chooses the face, so that every
// origin leaving there keeps its stepped coordinates within a voxel of the
// volume (ext: largest extent) and moves into the octant whose field is read:
// bu, cu say whether that lies upward along the stepped axes.  (A component of
// exactly zero can have a delta of either sign: the angles of a direction
// without an x component are those of one 0.001 off, and the octant is the
// zero's sign bit.)  A NaN fails its comparison.  scale: 65536 / the largest
// move of a step along the three axes, rounded down.
__device__ __forceinline__ bool exit_usable(const RayRule* __restrict__ rr, int axis,
                                            const AxisExit& e, bool bu, bool cu, int ext,
                                            int& scale) {
  const int b = axis == 0 ? 1 : 0, c = axis == 2 ? 1 : 2;
  const double sg = rr->neg ? -1.0 : 1.0;
  const double ea = __builtin_fabs(rr->dir[axis]), eb = sg * rr->dir[b], ec = sg * rr->dir[c];
  const double db = rr->d[e.face][b], dc = rr->d[e.face][c];
  const double mb = __builtin_fabs(db), mc = __builtin_fabs(dc);
  const double slack = 0.25 / (double)(ext + 1) * ea;
  const float most = (float)(mb > mc ? mb : mc);
  scale = most > 0.99999f ? (int)(65536.0f * 0.9999f / most) : 65536;
  if (mb <= 1.0 && mc <= 1.0) scale = 65536;
  return (rr->meta[e.face] & kMetaValid) && ea >= 0x1p-500 && ea <= 0x1p500 && mb <= 0x1p20 &&
         mc <= 0x1p20 && __builtin_fabs(db * ea - eb) <= slack &&
         __builtin_fabs(dc * ea - ec) <= slack && (db == 0.0 || (db > 0.0) == bu) &&
         (dc == 0.0 || (dc > 0.0) == cu);
}

// Offset of a stepped axis at m = RN(inc * d); `near` when some origin's
// c + m could round onto the boundary above.
__device__ __forceinline__ int step_offset(double m, bool round, bool& near) {
  const double f = __builtin_floor(m);
  const double r = m - f;                       // exact; 1 for a tiny negative m
  const double gap = round ? 0.5 - r : 1.0 - r; // to the boundary above (or past it)
  near = near || (round ? (gap > 0.0 && gap < 0x1p-40) : gap < 0x1p-40);
  return (int)f + ((round && r >= 0.5) ? 1 : 0);
}

// (m & a) | (~m & b), m uniform
__device__ __forceinline__ unsigned bit_select(unsigned m, unsigned a, unsigned b) {
  unsigned r;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "s"(m), "v"(a), "v"(b));
  return r;
}

// How a walk reads its field.  Words: a position, or a table's entry, as words
// whose sums are the position after a step.
struct VoxelField {
  struct alignas(8) Words { unsigned x, y; };   // x; y and z
  static constexpr int kVox = kSkipVox;
  static constexpr bool kCells = false;
  __amdgpu_buffer_rsrc_t rsrc;

  static __device__ __forceinline__ Words offset(int oz, int oy, int ox, const SkipArgs& k) {
    const unsigned gap_y = (((1u << k.hx) - 1u) << 7);   // x's high bits: y's carry runs through
    return Words{dilate_x(ox) | 0x78u, (dilate_y(oy, k.hx) | gap_y) + (unsigned)(oz * k.zs)};
  }
  __device__ __forceinline__ void aim(const SkipArgs& k, int oct) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(k.field + (long long)oct * k.oct_bytes),
                                             (short)0, (int)k.oct_bytes, 0x00020000);
  }
  static __device__ __forceinline__ Words origin(const int4& q) {
    return Words{(unsigned)q.z, (unsigned)q.w};
  }
  // the label at origin + w and 8 x the steps it holds for
  __device__ __forceinline__ void read(const SkipArgs& k, const Words& at, const Words& w, int& lab,
                                       int& s8) const {
    const unsigned mx = 7u | (((1u << k.hx) - 1u) << 7);
    const unsigned off = bit_select(mx, at.x + w.x, at.y + w.y);
    const int b = __builtin_amdgcn_raw_buffer_load_b8(rsrc, (int)off, 0, 0);
    lab = b & 7;
    s8 = b & 0xf8;
  }
  static __device__ __forceinline__ int bytes(int s8) { return s8; }
  static __device__ __forceinline__ int steps8(int bytes) { return bytes; }
};

// The field by cells of 4 x 4 x 4 voxels, for volumes larger than the caches:
// a byte per cell and octant (label or 7 where the cell's voxels differ; in
// bits 3-7 the side, in cells, of the cube of one label that starts at the
// cell), and the voxels' labels at 2 or 4 bits for cells of 7. A voxel at
// offset o (its largest over the axes, counted in the ray's direction) of a
// cell that starts a cube of k cells holds for 4 k - o steps.
//
// One address serves both: bit by bit from the lowest, x0 x1 y0 y1 z0 z1 within
// the cell, then x2 y2 z2 x3 y3 z3 x4, then x's high bits, y's, and z's by
// multiples of a tile plane. Its cell is the address / 64, the label its
// 2-bit or 4-bit element. A 128-byte line is 32 x 16 x 16 voxels of the
// field and 8 x 8 x 8 2-bit labels. x, y and z step in a word each, with the
// others' bits as gaps.
//
// 1000x1000x800: 13.6 MB per octant in place of 828 MB, 28 gathers per ray and
// 8 of single labels (the voxel field: 19).  100,000 voxels, 1,500 reflections:
// 153 ms stepping through bricks, 53.9 ms by the voxel field, 28.8 ms by cells;
// bound by the latency of dependent gathers (VALU and texture addresser both
// half busy): the tables' 26 KB of LDS leave four workgroups per CU.
struct CellField {
  struct Words { unsigned x, y, z; };
  static constexpr int kVox = 2;
  static constexpr bool kCells = true;
  static constexpr unsigned kMaskX = 0x1243u, kMaskY = 0x048cu, kMaskZ = 0x0930u;
  unsigned mx, tiles, flip;
  int shift;
  __amdgpu_buffer_rsrc_t rsrc, fine;

  static __host__ __device__ __forceinline__ Words dilate(int z, int y, int x, int hx) {
    Words w;
    w.x = (unsigned)((x & 3) | (x & 4) << 4 | (x & 8) << 6 | (x & 16) << 8) +
          ((unsigned)(x >> 5) << 13);
    w.y = (unsigned)((y & 3) << 2 | (y & 4) << 5 | (y & 8) << 7) +
          ((unsigned)(y >> 4) << (13 + hx));
    w.z = (unsigned)((z & 3) << 4 | (z & 4) << 6 | (z & 8) << 8) + ((unsigned)(z >> 4) << 12);
    return w;
  }
  static __host__ __device__ __forceinline__ unsigned merge(const Words& w, unsigned mx,
                                                            unsigned tiles) {
    const unsigned xy = (w.x & mx) | (w.y & ~mx);
    return ((w.z & kMaskZ) | (xy & ~kMaskZ)) + ((w.z >> 12) * tiles << 13);
  }
  static __host__ __device__ __forceinline__ unsigned x_mask(int hx) {
    return kMaskX | (((1u << hx) - 1u) << 13);
  }

  static __device__ __forceinline__ Words offset(int oz, int oy, int ox, const SkipArgs& k) {
    Words w = dilate(oz, oy, ox, k.hx);      // gaps of ones: carries run through
    w.x |= 0x1fffu & ~kMaskX;
    w.y |= ((1u << (13 + k.hx)) - 1u) & ~kMaskY;
    w.z |= 0x0fffu & ~kMaskZ;
    return w;
  }
  __device__ __forceinline__ void aim(const SkipArgs& k, int oct) {
    mx = x_mask(k.hx);
    tiles = (unsigned)k.zs;
    shift = k.fine_shift;
    flip = (oct & 1 ? 3u : 0u) | (oct & 2 ? 12u : 0u) | (oct & 4 ? 48u : 0u);
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(k.field + (long long)oct * k.oct_bytes),
                                             (short)0, (int)k.oct_bytes, 0x00020000);
    fine = __builtin_amdgcn_make_buffer_rsrc((void*)k.fine, (short)0, (int)k.fine_bytes,
                                             0x00020000);
  }
  static __device__ __forceinline__ Words origin(const int4& q) {
    const int z = q.x & 0xffff;
    Words w;
    w.x = (unsigned)q.z;
    w.y = (unsigned)q.w;
    w.z = dilate(z + 1, 0, 0, 0).z;
    return w;
  }
  __device__ __forceinline__ void read(const SkipArgs&, const Words& at, const Words& w, int& lab,
                                       int& s8) const {
    const unsigned xy = bit_select(mx, at.x + w.x, at.y + w.y);
    const unsigned zw = at.z + w.z;
    const unsigned v = bit_select(kMaskZ, zw, xy) + (__umul24(zw >> 12, tiles) << 13);
    const int b = __builtin_amdgcn_raw_buffer_load_b8(rsrc, (int)(v >> 6), 0, 0);
    const unsigned g = v ^ flip;
    const unsigned o = max(g & 3u, max((g >> 2) & 3u, (g >> 4) & 3u));
    lab = b & 7;
    s8 = ((b & 0xf8) << 2) - (int)(o << 3);
    if (lab == 7) {
      const int c = __builtin_amdgcn_raw_buffer_load_b8(fine, (int)(v >> shift), 0, 0);
      lab = shift == 2 ? (c >> ((v & 3u) << 1)) & 3 : (c >> ((v & 1u) << 2)) & 7;
      s8 = 8;
    }
    s8 = lab == 0 ? 8 : s8;
  }
  // bytes of the table for 8 x steps, and back
  static __device__ __forceinline__ int bytes(int s8) { return s8 + (s8 >> 1); }
  static __device__ __forceinline__ int steps8(int bytes) { return bytes * 2 / 3; }
};
static_assert(sizeof(CellField::Words) == 12, "table entry");

// Cells of the padded volume with a shell of zeros (the layout the field
// kernels read), and every cell's labels at 2 or 4 bits.  One thread per cell.
struct CellShape {
  int Z, Y, X;                 // cells
  int hx, tiles;               // bits of the x tile index, tiles per z plane
  int shift;                   // fine labels: 2^shift to a byte
};

__global__ void cell_label_kernel(const uint8_t* __restrict__ vol, int Z, int Y, int X,
                                  CellShape s, uint8_t* __restrict__ cells,
                                  uint32_t* __restrict__ fine) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)(s.Z + 2) * (s.Y + 2) * (s.X + 2)) return;
  const int cx = (int)(i % (s.X + 2)) - 1;
  const long long u = i / (s.X + 2);
  const int cy = (int)(u % (s.Y + 2)) - 1, cz = (int)(u / (s.Y + 2)) - 1;
  if (cx < 0 || cy < 0 || cz < 0 || cx >= s.X || cy >= s.Y || cz >= s.Z) {
    cells[i] = 0;
    return;
  }
  const int bits = 4 >> (s.shift - 1);
  int first = -1;
  bool same = true;
  const CellField::Words w = CellField::dilate(4 * cz, 4 * cy, 4 * cx, s.hx);
  const unsigned at = CellField::merge(w, CellField::x_mask(s.hx), (unsigned)s.tiles);
  uint32_t* const out = fine + ((at >> s.shift) >> 2);
  uint32_t word = 0;
  int have = 0;
  for (int v = 0; v < 64; ++v) {
    const int l = padded_label(vol, Z, Y, X, 4 * cz + (v >> 4), 4 * cy + ((v >> 2) & 3),
                               4 * cx + (v & 3));
    if (first < 0) first = l;
    same = same && l == first;
    word |= (uint32_t)l << have;
    have += bits;
    if (have == 32) {
      out[v * bits / 32] = word;
      word = 0;
      have = 0;
    }
  }
  cells[i] = (uint8_t)(same ? first : 7);
}

// All eight octants of a cell from the bit planes (field_pack_kernel's rule).
__global__ void cell_pack_kernel(const uint8_t* __restrict__ cells, CellShape s, int wx,
                                 const uint32_t* __restrict__ planes, long long plane_words,
                                 uint8_t* __restrict__ field, long long oct_bytes) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)s.Z * s.Y * s.X) return;
  const int cx = (int)(i % s.X) + 1;           // in the padded grid
  const long long u = i / s.X;
  const int cy = (int)(u % s.Y) + 1, cz = (int)(u / s.Y) + 1;
  const int label = cells[((long long)cz * (s.Y + 2) + cy) * (s.X + 2) + cx];
  const CellField::Words w = CellField::dilate(4 * (cz - 1), 4 * (cy - 1), 4 * (cx - 1), s.hx);
  const unsigned at =
      CellField::merge(w, CellField::x_mask(s.hx), (unsigned)s.tiles) >> 6;
  for (int o = 0; o < 8; ++o) {
    int n = label == 7 ? 0 : 1;
    for (int l = 0; n && label && l < kLevels; ++l) {   // label 0 ends a ray: no cube counts
      const int k = kLevelSide[l];
      const int qz = (o & 4) ? max(cz - k, 0) : cz;
      const int qy = (o & 2) ? max(cy - k, 0) : cy;
      const int qx = (o & 1) ? max(cx - k, 0) : cx;
      const uint32_t word = planes[l * plane_words + ((long long)qz * (s.Y + 2) + qy) * wx +
                                   (qx >> 5)];
      if (!((word >> (qx & 31)) & 1u)) break;  // higher levels hold larger cubes
      n = k + 1;
    }
    field[(long long)o * oct_bytes + at] = (uint8_t)(label | (n << 3));
  }
}
// One ray direction in a workgroup: its exits, field and table.  Args: the
// volume's extents Z, Y, X, voxel edges vs and coefficients mu.
template <class Field>
struct SkipRay {
  typedef typename Field::Words Words;
  AxisExit ez, ey, ex;
  Field f;
  float iz, iy, ix;            // 1 / |direction|
  int sz, sy, sx, oz, oy, ox;  // distance to the exit plane along an axis: o + s * c

  // Builds the tables; every thread of the workgroup, behind a barrier after
  // the last reader of the previous ray's.
  template <class Args>
  __device__ __forceinline__ SkipRay(const RayRule* __restrict__ rr, const Args& a,
                                     const SkipArgs& k, AxisLds* axes, Words* tbl)
      : ez(rr, 0), ey(rr, 1), ex(rr, 2) {
    const int tid = (int)threadIdx.x;
    if (tid < 3) {
      const AxisExit e = tid == 0 ? ez : tid == 1 ? ey : ex;
      const double* d = rr->d[e.face];
      AxisLds& A = axes[tid];
      A.at = k.at[tid] * (int)sizeof(Words);
      A.near = exit_usable(rr, tid, e, tid == 0 ? ey.up : ez.up, tid == 2 ? ey.up : ex.up,
                           max(a.Z, max(a.Y, a.X)), A.scale) ? 0x7fffffff
               : (rr->meta[e.face] & kMetaValid) ? 0 : -1;
      A.add = e.add;
      A.hb = (tid == 0 ? a.Y : a.Z) - 1;
      A.hc = (tid == 2 ? a.Y : a.X) - 1;
      A.face = e.face;
      A.up = e.up ? 1 : 0;
      A.db = d[tid == 0 ? 1 : 0];
      A.dc = d[tid == 2 ? 1 : 2];
      A.vb = a.vs[tid == 0 ? 1 : 0];
      A.vc = a.vs[tid == 2 ? 1 : 2];
      A.vp = a.vs[tid];
      A.bias = e.round ? kRoundBias : 0.0;
    }
    __syncthreads();
    // offsets of the increments that any listed voxel takes
    auto build = [&](const AxisExit& e, int axis, int ext) {
      const int n = (e.up ? ext - k.lo[axis] : k.hi[axis]) + e.add;
      Words* const out = tbl + k.at[axis];
      const double* d = rr->d[e.face];
      const double db = axis == 0 ? d[1] : d[0], dc = axis == 2 ? d[1] : d[2];
      int first = 0x7fffffff;
      for (int inc = tid; inc < n; inc += kBlock) {
        bool near = false;
        const int op = e.up ? inc : -inc;
        const int ob = step_offset((double)inc * db, e.round, near);
        const int oc = step_offset((double)inc * dc, e.round, near);
        const int oz = axis == 0 ? op : ob;
        const int oy = axis == 0 ? ob : axis == 1 ? op : oc;
        const int ox = axis == 2 ? op : oc;
        out[inc] = Field::offset(oz, oy, ox, k);
        if (near) first = min(first, inc);
      }
      if (first != 0x7fffffff) atomicMin(&axes[axis].near, first);
    };
    build(ez, 0, a.Z);
    build(ey, 1, a.Y);
    build(ex, 2, a.X);
    __syncthreads();
    const int oct = (ez.up ? 0 : 4) | (ey.up ? 0 : 2) | (ex.up ? 0 : 1);
    f.aim(k, oct);
    iz = (float)__builtin_fabs(rr->d[0][3]);
    iy = (float)__builtin_fabs(rr->d[1][3]);
    ix = (float)__builtin_fabs(rr->d[2][3]);
    sz = ez.up ? -1 : 1;
    sy = ey.up ? -1 : 1;
    sx = ex.up ? -1 : 1;
    oz = ez.up ? a.Z : 0;
    oy = ey.up ? a.Y : 0;
    ox = ex.up ? a.X : 0;
  }

  // mu * length of one voxel's ray; where the walk does not cover it, kRayRedo
  // in err (in LDS: hardly a ray needs it) and 0, where the reference aborts the
  // stepping kernel's error and NaN.  col: this lane's step counters (zero
  // before and after).
  template <class Args>
  __device__ __forceinline__ double trace(const RayRule* __restrict__ rr, const int4 q,
                                          const Args& a, const SkipArgs& k, const AxisLds* axes,
                                          const Words* tbl, uint32_t* col, unsigned* err,
                                          unsigned& steps) const {
    double r = 0.0;
    const int z = q.x & 0xffff, y = (int)((unsigned)q.x >> 16), x = q.y;
    // cube_face by FP32 products with the reciprocals; FP64 quotients
    // decide where two planes are closer than the products' rounding
    const int kz = mad24(z, sz, oz), ky = mad24(y, sy, oy), kx = mad24(x, sx, ox);
    const float tz = (float)kz * iz, ty = (float)ky * iy, tx = (float)kx * ix;
    const bool z_first = tz < ty;
    const float lo = z_first ? tz : ty, hi = z_first ? ty : tz;
    const bool x_first = tx < lo;
    const float t0 = x_first ? tx : lo;
    const float t1 = x_first ? lo : (hi < tx ? hi : tx);
    int p = x_first ? 2 : z_first ? 0 : 1;
    bool use = true;
    if (!(t1 > t0 * 1.00001f) || min(z, min(y, x)) == 0) {
      const int face = exit_face<true>(z, y, x, rr->dir[0], rr->dir[1], rr->dir[2],
                                       rr->d[0][3], rr->d[1][3], rr->d[2][3], a.Z, a.Y, a.X,
                                       rr->neg != 0);
      p = (face == 2 || face == 3) ? 0 : (face == 4 || face == 5) ? 1 : 2;
      use = face - 1 == axes[p].face;
      // a voxel on the lower plane that the reference finds first, at distance 0
      // also for a ray that leaves it: one step, of length 0, whatever the deltas
      const bool lower = face == 2 || face == 4 || face == 6;
      if (lower && (p == 0 ? z : p == 1 ? y : x) == 0) {
        if (rr->meta[face - 1] & kMetaValid) {
          ++steps;
          return 0.0;
        }
        atomicOr(err, ANACOR_RAY_ERR_ASSERT);
        return __builtin_nan("");
      }
    }
    const AxisLds& A = axes[p];
    const int kp = p == 0 ? kz : p == 1 ? ky : kx;
    const int limit = kp + A.add;
    if (!use || limit > A.near) {
      const bool abort = use && A.near < 0;
      atomicOr(err, abort ? ANACOR_RAY_ERR_ASSERT : kRayRedo);
      if (abort) r = __builtin_nan("");
    } else {
      const int scale = A.scale;
      const Words at = Field::origin(q);
      const char* t = (const char*)tbl + A.at;      // the increment's entry
      const char* const end = t + limit * (int)sizeof(Words);
      int lab;
      auto walk = [&](bool unit) {
        do {
          int s8;                                   // 8 x steps the label holds for
          f.read(k, at, *(const Words*)t, lab, s8);
          if (!unit) s8 = ((int)(__umul24((unsigned)(s8 - 8), (unsigned)scale) >> 16) & ~7) + 8;
          atomicAdd(col + lab * kBlock, (unsigned)s8);
          t += Field::bytes(s8);
        } while (lab != 0 && t < end);
      };
      // a wave whose rays all step at most one voxel per axis (most)
      // skips without scaling
      if (__all(scale == 65536)) walk(true);
      else walk(false);
      // a last label past the end counted the steps beyond it too
      const int over = Field::steps8((int)(t - end));
      const int len = lab == 0 ? limit + (over >> 3) - 1 : limit;
      steps += (unsigned)len;
      const int n8 = max(lab == 0 ? 0 : over, 0);
      // sum of mu over the steps, label by label
      double W = a.mu[0] * (double)(int)(col[1 * kBlock] - (lab == 1 ? n8 : 0));
      W = __builtin_fma(a.mu[1], (double)(int)(col[2 * kBlock] - (lab == 2 ? n8 : 0)), W);
      W = __builtin_fma(a.mu[2], (double)(int)(col[3 * kBlock] - (lab == 3 ? n8 : 0)), W);
      W = __builtin_fma(a.mu[3], (double)(int)(col[4 * kBlock] - (lab == 4 ? n8 : 0)), W);
#pragma unroll
      for (int l = 1; l < 5; ++l) col[l * kBlock] = 0;
      if (len > 1) {
        const int last = len - 1;
        const double D = (double)last;
        const int cb = p == 0 ? y : z, cc = p == 2 ? y : x;
        const int ib = axis_index<false>((double)cb, D, A.db, A.bias, A.hb);
        const int ic = axis_index<false>((double)cc, D, A.dc, A.bias, A.hc);
        const int dp = min(last, kp - A.up);
        const double b_ = (double)(ib - cb) * A.vb;
        const double c_ = (double)(ic - cc) * A.vc;
        const double p_ = (double)dp * A.vp;
        r = ray_weight(__builtin_fma(b_, b_, __builtin_fma(c_, c_, p_ * p_)), W * 0.125, D,
                       [](double v) { return __builtin_amdgcn_rsq(v); },
                       [](double v) { return __builtin_amdgcn_rcp(v); });
      }
    }
    return r;
  }
};

template <class Field, bool F64>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(Field::kCells ? 4 : F64 ? 6 : 8)))
void skip_kernel(TraceArgs a, SkipArgs k) {
  extern __shared__ uint2 tables[];             // offsets by increment: z, y, x exits
  typename Field::Words* const tbl = (typename Field::Words*)tables;
  constexpr int kVox = Field::kVox;
  __shared__ uint32_t hist[5 * kBlock];         // 8 x steps per label, one column per lane
  __shared__ AxisLds axes[3];
  __shared__ double incident[kVox * kBlock];  // the first ray's exponent per voxel
  __shared__ ReduceLds red;
  __shared__ unsigned err;

  const int lb = xcd_logical_block((int)blockIdx.x, (int)gridDim.x);
  if (lb >= a.n_blocks) return;
  int pos, tile;
  block_work(lb, a.tiles, a.R, a.group, pos, tile);
  pos += a.pos0;
  const int refl = a.order[pos];
  const ReflRule* __restrict__ rule = a.rules + refl;
  const int tid = (int)threadIdx.x;
  uint32_t* const col = hist + tid;
#pragma unroll
  for (int l = 1; l < 5; ++l) col[l * kBlock] = 0;
  if (tid == 0) err = 0;
  TileAcc acc = {0.f, 0.f, 0.0, 0ull, 0u};
  unsigned steps = 0;
  const int v_begin = tile * a.vox_per_tile;
  const int v_end = min(a.N, v_begin + a.vox_per_tile);

  for (int s0 = v_begin; s0 < v_end; s0 += kVox * kBlock) {
#pragma unroll 1
    for (int ray = 0; ray < 2; ++ray) {
      const RayRule* __restrict__ rr = &rule->ray[ray];
      __syncthreads();                          // the table's last readers are done
      if (__builtin_amdgcn_readfirstlane((int)err) & kRayRedo) {   // traced again anyway
        s0 = v_end;
        break;
      }
      const SkipRay<Field> walk(rr, a, k, axes, tbl);
      // where the first ray aborts there is no second one (its voxels hold NaN)
      const bool aborts = ray == 1 && __builtin_amdgcn_readfirstlane((int)err) != 0;
      const int s1 = min(v_end, s0 + kVox * kBlock);
#pragma unroll 1
      for (int v = s0 + tid; v < s1; v += kBlock) {
        if (aborts) {
          int w = v - s0;                         // its own address: no register across trace()
          asm volatile("" : "+v"(w));
          if (incident[w] != incident[w]) continue;
        }
        double r = walk.trace(rr, k.vox[v], a, k, axes, tbl, col, &err, steps);
        double* const first = incident + (v - s0);
        if (ray == 0) {
          *first = r;
          continue;
        }
        r += *first;
        if (F64) {
          acc.acc64 += a.is_exp ? exp(-r) : r;
        } else {
          const float val = a.is_exp ? exp_neg(r) : (float)r;
          const float yv = val - acc.kc;
          const float t = acc.ks + yv;
          acc.kc = (t - acc.ks) - yv;
          acc.ks = t;
        }
      }
    }
  }
  acc.steps = steps;
  const int slot = pos * a.tiles + tile;
  reduce_tile<F64, false>(acc, red, &a.err[refl], a.steps + refl, a.partial32 + slot,
                          a.partial64 + slot);
  if (tid == 0 && err) {                        // behind reduce_tile's barrier
    // a second ray that the walk did not look at behind an aborting first one may
    // have no exit face, which is then the error to report
    const double* const d = rule->ray[1].dir;
    const bool face = __builtin_isfinite(d[0]) && __builtin_isfinite(d[1]) &&
                      __builtin_isfinite(d[2]);
    atomicOr(&a.err[refl], face ? err : err | kRayRedo);
  }
}

// The absorption map (grid_map_kernel) by the skip walk: one direction per
// workgroup and tile, whose table serves every voxel of the tile.  A direction
// that the walk does not cover is marked and mapped by the stepping kernel.
// 150x201x187, 4,000 voxels, 7,200 directions: 3.97 ms stepping, 1.22 ms so,
// marked directions included; bound as skip_kernel is.
template <class Field>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(Field::kCells ? 4 : 6)))
void skip_map_kernel(GridArgs a, SkipArgs k) {
  extern __shared__ uint2 tables[];
  typename Field::Words* const tbl = (typename Field::Words*)tables;
  __shared__ uint32_t hist[5 * kBlock];
  __shared__ AxisLds axes[3];
  __shared__ unsigned err;
  const int lb = xcd_logical_block((int)blockIdx.x, (int)gridDim.x);
  if (lb >= a.n_blocks) return;
  const int d = lb / a.tiles;
  const int tile = lb - d * a.tiles;
  uint32_t* const col = hist + threadIdx.x;
#pragma unroll
  for (int l = 1; l < 5; ++l) col[l * kBlock] = 0;
  const RayRule* __restrict__ rr = a.rays + d;
  if (threadIdx.x == 0) err = 0;
  const SkipRay<Field> walk(rr, a, k, axes, tbl);
  unsigned steps = 0;
  const int v_end = min(a.N, (tile + 1) * a.vox_per_tile);
#pragma unroll 1
  for (int v = tile * a.vox_per_tile + (int)threadIdx.x; v < v_end; v += kBlock) {
    const double r = walk.trace(rr, k.vox[v], a, k, axes, tbl, col, &err, steps);
    a.map[(size_t)d * a.N + k.index[v]] = (float)(a.is_exp ? exp(-r) : r);
  }
  __syncthreads();
  if (threadIdx.x == 0 && err) atomicOr(&a.err[d], err);
}
