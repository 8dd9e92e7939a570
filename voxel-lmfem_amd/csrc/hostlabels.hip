// Host passes over label and orientation arrays (no device work), cut into
// pieces on a few threads: a label array of 256^3 voxels is read once at
// memory speed instead of by several single-threaded NumPy passes.
#include "vxl_internal.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <thread>

namespace vxl {
namespace {

constexpr int64_t kPiece = 1 << 18;  // entries per piece; fewer than two pieces run on the calling thread
// Widest label range a piece marks in a table of its own.  Labels in no order, 8 threads:
// 96^3 voxels of 200 labels 0.4 ms, 48^3 of 2 labels 0.09; marking a shared table
// wherever the label changes took 7.9 and 0.8 ms (the threads write the same cache
// lines, and the branch is a coin toss), bincount over pieces 1.8 and 0.3.
constexpr int64_t kOwnTable = 1 << 14;

// f(piece) for every piece, on at most `workers` threads.
template <typename F>
void for_pieces(int64_t pieces, int workers, F&& f) {
  const int nt = int(std::min<int64_t>(std::max(1, workers), pieces));
  std::atomic<int64_t> next{0};
  auto run = [&]() {
    for (int64_t k = next.fetch_add(1); k < pieces; k = next.fetch_add(1)) f(k);
  };
  std::vector<std::thread> pool;
  for (int t = 1; t < nt; ++t) {
    try {
      pool.emplace_back(run);
    } catch (...) {
      break;  // no more threads: the ones there are do the work
    }
  }
  run();
  for (auto& t : pool) t.join();
}

template <typename F>
int by_label_type(int bytes, int is_signed, F&& f) {
  switch (bytes * 2 + (is_signed ? 1 : 0)) {
    case 2: return f(uint8_t());
    case 3: return f(int8_t());
    case 4: return f(uint16_t());
    case 5: return f(int16_t());
    case 8: return f(uint32_t());
    case 9: return f(int32_t());
    case 17: return f(int64_t());
  }
  return fail("unsupported label type");
}

inline int64_t pieces_of(int64_t count) { return (count + kPiece - 1) / kPiece; }

}  // namespace
}  // namespace vxl

using namespace vxl;

extern "C" {

int vxl_host_label_range(const void* labels, int bytes, int is_signed, int64_t count, int workers, long long* lo,
                         long long* hi) {
  if (!labels || count < 1 || !lo || !hi) return fail("vxl_host_label_range: invalid arguments");
  return by_label_type(bytes, is_signed, [&](auto tag) -> int {
    using L = decltype(tag);
    const L* p = static_cast<const L*>(labels);
    const int64_t n = pieces_of(count);
    std::vector<L> mn(n), mx(n);
    for_pieces(n, workers, [&](int64_t k) {
      const int64_t a = k * kPiece, b = std::min(count, a + kPiece);
      L lo1 = p[a], hi1 = p[a];
      for (int64_t i = a; i < b; ++i) {
        lo1 = std::min(lo1, p[i]);
        hi1 = std::max(hi1, p[i]);
      }
      mn[k] = lo1;
      mx[k] = hi1;
    });
    *lo = static_cast<long long>(*std::min_element(mn.begin(), mn.end()));
    *hi = static_cast<long long>(*std::max_element(mx.begin(), mx.end()));
    return VXL_OK;
  });
}

int vxl_host_label_mark(const void* labels, int bytes, int is_signed, int64_t count, int workers, long long lo,
                        int64_t span, uint8_t* present) {
  if (!labels || count < 1 || span < 1 || !present) return fail("vxl_host_label_mark: invalid arguments");
  return by_label_type(bytes, is_signed, [&](auto tag) -> int {
    using L = decltype(tag);
    const L* p = static_cast<const L*>(labels);
    std::atomic<bool> outside{false};
    for_pieces(pieces_of(count), workers, [&](int64_t k) {
      const int64_t a = k * kPiece, b = std::min(count, a + kPiece);
      bool bad = false;
      if (span <= kOwnTable) {
        // A table of the piece's own, one store per voxel: no branch on the labels, and no
        // cache line written by several threads, until the tables are joined.
        uint8_t own[kOwnTable];
        std::fill(own, own + span, uint8_t(0));
        for (int64_t i = a; i < b; ++i) {
          const uint64_t at = uint64_t(int64_t(p[i])) - uint64_t(lo);
          if (at < uint64_t(span))
            own[at] = 1;
          else
            bad = true;
        }
        for (int64_t l = 0; l < span; ++l)
          if (own[l] && !__atomic_load_n(present + l, __ATOMIC_RELAXED))
            __atomic_store_n(present + l, uint8_t(1), __ATOMIC_RELAXED);
      } else {
        // Wide ranges: the shared table, looked up where the label changes and written only
        // where an entry is not set yet.
        L last = p[a];
        auto mark = [&](L v) {
          const uint64_t at = uint64_t(int64_t(v)) - uint64_t(lo);
          if (at >= uint64_t(span))
            bad = true;
          else if (!__atomic_load_n(present + at, __ATOMIC_RELAXED))
            __atomic_store_n(present + at, uint8_t(1), __ATOMIC_RELAXED);
        };
        mark(last);
        for (int64_t i = a + 1; i < b; ++i)
          if (p[i] != last) mark(last = p[i]);
      }
      if (bad) outside = true;
    });
    return outside ? fail("vxl_host_label_mark: label outside the range") : VXL_OK;
  });
}

int vxl_host_label_pack(const void* labels, int bytes, int is_signed, int64_t count, int workers, long long lo,
                        int out_bytes, void* out) {
  if (!labels || count < 1 || !out || (out_bytes != 1 && out_bytes != 2))
    return fail("vxl_host_label_pack: invalid arguments");
  return by_label_type(bytes, is_signed, [&](auto tag) -> int {
    using L = decltype(tag);
    const L* p = static_cast<const L*>(labels);
    for_pieces(pieces_of(count), workers, [&](int64_t k) {
      const int64_t a = k * kPiece, b = std::min(count, a + kPiece);
      const L base = static_cast<L>(lo);
      if (out_bytes == 1) {
        uint8_t* o = static_cast<uint8_t*>(out);
        for (int64_t i = a; i < b; ++i) o[i] = static_cast<uint8_t>(p[i] - base);
      } else {
        uint16_t* o = static_cast<uint16_t*>(out);
        for (int64_t i = a; i < b; ++i) o[i] = static_cast<uint16_t>(p[i] - base);
      }
    });
    return VXL_OK;
  });
}

int vxl_host_find_label(const void* labels, int bytes, int is_signed, int64_t count, int workers, long long label,
                        int64_t capacity, int64_t* out, int64_t* found) {
  if (!labels || count < 1 || !found || (capacity > 0 && !out)) return fail("vxl_host_find_label: invalid arguments");
  return by_label_type(bytes, is_signed, [&](auto tag) -> int {
    using L = decltype(tag);
    const L* p = static_cast<const L*>(labels);
    const L want = static_cast<L>(label);
    if (static_cast<long long>(want) != label) {  // not a value of this type
      *found = 0;
      return VXL_OK;
    }
    // Positions of the label in [a, b) to out[o ...], which holds those up to `end`: a group of
    // 32 without a match takes one compare in vector registers, the others write every
    // position over the next free entry, without a branch on the labels.  Returns the next o.
    auto collect = [&](int64_t a, int64_t b, int64_t o, int64_t end) {
      for (int64_t g = a; g < b && o < end; g += 32) {
        const int64_t e = std::min(b, g + 32);
        bool any = e - g < 32;
        if (!any)
          for (int j = 0; j < 32; ++j) any |= p[g + j] == want;
        if (!any) continue;
        for (int64_t i = g; i < e && o < end; ++i) {
          out[o] = i;
          o += p[i] == want;
        }
      }
      return o;
    };
    const int64_t n = pieces_of(count);
    if (n == 1 && capacity >= count) {  // room for every voxel: no count first
      *found = collect(0, count, 0, count);
      return VXL_OK;
    }
    std::vector<int64_t> start(n + 1, 0);
    for_pieces(n, workers, [&](int64_t k) {
      const int64_t a = k * kPiece, b = std::min(count, a + kPiece);
      start[k + 1] = std::count(p + a, p + b, want);
    });
    for (int64_t k = 0; k < n; ++k) start[k + 1] += start[k];
    *found = start[n];
    if (start[n] > capacity) return VXL_OK;  // the caller asks again with room
    for_pieces(n, workers, [&](int64_t k) {
      collect(k * kPiece, std::min(count, (k + 1) * kPiece), start[k], start[k + 1]);
    });
    return VXL_OK;
  });
}

int vxl_host_check_axes(const double* axis1, const double* axis2, const int64_t* voxels, int64_t count, int64_t piece,
                        int workers, double* out1, double* out2, int* code) {
  if (!axis1 || !axis2 || !voxels || count < 1 || piece < 1 || !out1 || !out2 || !code)
    return fail("vxl_host_check_axes: invalid arguments");
  const int64_t n = (count + piece - 1) / piece;
  std::vector<int> bad(n, 0);
  for_pieces(n, workers, [&](int64_t k) {
    bool f1 = false, f2 = false, zero = false, line = false;
    const int64_t first = k * piece, last = std::min(count, first + piece);
    for (int64_t e = first; e < last; ++e) {
      const double* a = axis1 + 3 * voxels[e];
      const double* b = axis2 + 3 * voxels[e];
      const double a0 = a[0], a1 = a[1], a2 = a[2], b0 = b[0], b1 = b[1], b2 = b[2];
      out1[3 * e] = a0;
      out1[3 * e + 1] = a1;
      out1[3 * e + 2] = a2;
      out2[3 * e] = b0;
      out2[3 * e + 1] = b1;
      out2[3 * e + 2] = b2;
      f1 |= !(std::isfinite(a0) && std::isfinite(a1) && std::isfinite(a2));
      f2 |= !(std::isfinite(b0) && std::isfinite(b1) && std::isfinite(b2));
      const double na = std::sqrt(a0 * a0 + a1 * a1 + a2 * a2), nb = std::sqrt(b0 * b0 + b1 * b1 + b2 * b2);
      zero |= na <= 0 || nb <= 0;
      const double x0 = a0 / na, x1 = a1 / na, x2 = a2 / na, y0 = b0 / nb, y1 = b1 / nb, y2 = b2 / nb;
      const double c0 = x1 * y2 - x2 * y1, c1 = x2 * y0 - x0 * y2, c2 = x0 * y1 - x1 * y0;
      line |= std::sqrt(c0 * c0 + c1 * c1 + c2 * c2) <= 1e-12;
    }
    bad[k] = f1 || f2 ? 1 : zero ? 2 : line ? 3 : 0;
  });
  *code = 0;
  for (int64_t k = 0; k < n && !*code; ++k) *code = bad[k];
  return VXL_OK;
}

}  // extern "C"
