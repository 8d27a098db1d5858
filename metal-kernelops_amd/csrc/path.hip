// Four-path layout of the 2D selective scan (VMamba's ss2d) for gfx950.
//
// A (batch, rows, H, W) map is read along four paths; path k visits pixel pos_k(i)
// at step i of L = H * W:
//   k = 0: i                         row-major
//   k = 1: (i % H) * W + i / H       column-major: down each column, columns left to right
//   k = 2: L - 1 - i                 path 0 reversed
//   k = 3: pos_1(L - 1 - i)          path 1 reversed
// `stack` writes the four paths of every row in step order, (batch, 4 rows, L), the
// layout the 1-D scan kernels take (4x the channels, or 4x the groups of B/C); `merge`
// adds the four step-ordered slices back at each pixel, (s0 + s2) + (s1 + s3), the
// order of the reference's merge_paths (cv/path_scan.py:372-404).
//
// One lane per (batch, row, step) or (batch, row, pixel): the contiguous side is the
// one the lane index walks, the transposed paths gather with stride W (stack) or H
// (merge).  Every operand is L2-resident at the map sizes this layer sees, and a launch costs
// more than the copies: one launch takes up to kMaps maps (blockIdx.y), the four inputs of a
// 2D scan or its four gradients (1 x 96 x 56 x 56, 16 states: four stacks 4 x 5 us as launches
// of their own, 8 us together).  Element indices are 32-bit where every map allows it (a
// 64-bit division takes five times as many instructions, and an element needs six).
#include "common.hpp"
#include "io.hpp"

namespace mko {
namespace path {
namespace {

struct Geo {
  int64_t batch, rows, height, width, length, total;  // total = batch * rows * length
  int dtype;
  float scale;
};

constexpr int kMaps = MKO_PATH_MAPS;

struct Map {
  Geo g;
  const void* src;
  void* dst;
};
struct Maps {
  Map m[kMaps];
};

template <class I>
__global__ void __launch_bounds__(256) stack(Maps maps) {
  const Map& m = maps.m[blockIdx.y];
  const Geo& g = m.g;
  const I e = static_cast<I>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= static_cast<I>(g.total)) return;
  const I L = static_cast<I>(g.length), H = static_cast<I>(g.height), W = static_cast<I>(g.width);
  const I rows = static_cast<I>(g.rows);
  const I br = e / L, i = e - br * L;
  const I b = br / rows, r = br - b * rows;
  const I j = L - 1 - i;
  const I qi = i / H, qj = j / H;
  const I col = (i - qi * H) * W + qi;   // pos_1(i)
  const I rcol = (j - qj * H) * W + qj;  // pos_1(L - 1 - i)
  const int64_t in = static_cast<int64_t>(br) * g.length;
  const int64_t out = (static_cast<int64_t>(b) * 4 * g.rows + r) * g.length + i;
  const int64_t slice = g.rows * g.length;
  store_one(m.dst, g.dtype, out, g.scale * load_one(m.src, g.dtype, in + i));
  store_one(m.dst, g.dtype, out + slice, g.scale * load_one(m.src, g.dtype, in + col));
  store_one(m.dst, g.dtype, out + 2 * slice, g.scale * load_one(m.src, g.dtype, in + j));
  store_one(m.dst, g.dtype, out + 3 * slice, g.scale * load_one(m.src, g.dtype, in + rcol));
}

template <class I>
__global__ void __launch_bounds__(256) merge(Maps maps) {
  const Map& m = maps.m[blockIdx.y];
  const Geo& g = m.g;
  const I e = static_cast<I>(blockIdx.x) * 256 + threadIdx.x;
  if (e >= static_cast<I>(g.total)) return;
  const I L = static_cast<I>(g.length), H = static_cast<I>(g.height), W = static_cast<I>(g.width);
  const I rows = static_cast<I>(g.rows);
  const I br = e / L, pix = e - br * L;
  const I b = br / rows, r = br - b * rows;
  const I h = pix / W, w = pix - h * W;
  const I col = w * H + h;  // the step at which path 1 stands on pix
  const int64_t base = (static_cast<int64_t>(b) * 4 * g.rows + r) * g.length;
  const int64_t slice = g.rows * g.length;
  const float s0 = load_one(m.src, g.dtype, base + pix);
  const float s1 = load_one(m.src, g.dtype, base + slice + col);
  const float s2 = load_one(m.src, g.dtype, base + 2 * slice + (L - 1 - pix));
  const float s3 = load_one(m.src, g.dtype, base + 3 * slice + (L - 1 - col));
  store_one(m.dst, g.dtype, e, ((s0 + s2) + (s1 + s3)) * g.scale);
}

int make_geo(const mko_path_params* p, Geo* g, const char* what) {
  if (!p) {
    mko_set_error("%s: null parameters", what);
    return MKO_EINVAL;
  }
  if (p->batch < 0 || p->rows < 0 || p->height < 0 || p->width < 0) {
    mko_set_error("%s: negative extent", what);
    return MKO_EINVAL;
  }
  if (p->dtype != MKO_F32 && p->dtype != MKO_F16 && p->dtype != MKO_BF16) {
    mko_set_error("%s: unknown dtype %d", what, p->dtype);
    return MKO_EINVAL;
  }
  g->batch = p->batch;
  g->rows = p->rows;
  g->height = p->height;
  g->width = p->width;
  g->length = p->height * p->width;
  g->total = p->batch * p->rows * g->length;
  g->dtype = p->dtype;
  g->scale = p->scale;
  if (g->total > 0 && (!p->src || !p->dst)) {
    mko_set_error("%s: src and dst are required", what);
    return MKO_EINVAL;
  }
  if (g->total > (int64_t{1} << 40)) {
    mko_set_error("%s: %lld elements is beyond the supported size", what, static_cast<long long>(g->total));
    return MKO_EUNSUPPORTED;
  }
  return MKO_OK;
}

unsigned blocks(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

}  // namespace
}  // namespace path
}  // namespace mko

using namespace mko;

extern "C" size_t mko_sizeof_path_params(void) { return sizeof(mko_path_params); }

static int run(const mko_path_params* p, int count, void* stream, bool stacks) {
  const char* what = stacks ? "path_stack" : "path_merge";
  if (count < 0 || count > path::kMaps) {
    mko_set_error("%s: %d maps, at most %d run together", what, count, path::kMaps);
    return MKO_EINVAL;
  }
  path::Maps maps{};
  int n = 0;
  int64_t most = 0;
  for (int i = 0; i < count; ++i) {
    path::Map m{};
    const int st = path::make_geo(p ? p + i : nullptr, &m.g, what);
    if (st != MKO_OK) return st;
    if (m.g.total == 0) continue;
    m.src = p[i].src;
    m.dst = p[i].dst;
    if (m.g.total > most) most = m.g.total;
    maps.m[n++] = m;
  }
  if (n == 0) return MKO_OK;
  const dim3 grid(path::blocks(most), n);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool small = most < (int64_t{1} << 31);
  if (stacks && small) MKO_TIMED("path_stack", s, path::stack<uint32_t><<<grid, 256, 0, s>>>(maps));
  else if (stacks) MKO_TIMED("path_stack", s, path::stack<int64_t><<<grid, 256, 0, s>>>(maps));
  else if (small) MKO_TIMED("path_merge", s, path::merge<uint32_t><<<grid, 256, 0, s>>>(maps));
  else MKO_TIMED("path_merge", s, path::merge<int64_t><<<grid, 256, 0, s>>>(maps));
  return mko_check_launch(what);
}

extern "C" int mko_path_stack(const mko_path_params* p, void* stream) { return run(p, 1, stream, true); }

extern "C" int mko_path_merge(const mko_path_params* p, void* stream) { return run(p, 1, stream, false); }

extern "C" int mko_path_stack_many(const mko_path_params* p, int count, void* stream) {
  return run(p, count, stream, true);
}

extern "C" int mko_path_merge_many(const mko_path_params* p, int count, void* stream) {
  return run(p, count, stream, false);
}
