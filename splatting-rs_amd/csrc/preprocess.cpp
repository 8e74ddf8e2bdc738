// Image preprocessing of both crates on the device: the input-size rules
// (depthanything3-rs/src/preprocess.rs:22-45, mapanything-rs/src/preprocess.rs:16-63), the
// `image` crate's resize (image 0.25.10, Cargo.lock:2536-2539, imageops/sample.rs: resize,
// vertical_sample, horizontal_sample and the Triangle / CatmullRom / Lanczos3 kernels; the crate
// is not vendored, this restates its published algorithm), center crops and to_model_input
// (mapanything-rs/src/image_input.rs:195-216).
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <map>
#include <sched.h>
#include <thread>
#include <vector>

#include "ring_fill.h"
#include "runtime.h"

namespace splat {

namespace {

// Staging slots of the preprocessing (Context::staging_buffer).
enum { SLOT_SRC = 40, SLOT_A = 41, SLOT_B = 42, SLOT_TMP = 43, SLOT_ROWS = 44, SLOT_COLS = 45, SLOT_BATCH = 46,
       SLOT_FLAGS = 49, SLOT_SRC2 = 50 };

ResizeTaps upload_taps(Context& c, int slot, const ResizeTapsHost& t) {
  const size_t n = t.first.size(), nw = t.w.size();
  std::vector<char> buf(3 * n * sizeof(int) + nw * sizeof(float));
  std::memcpy(buf.data(), t.first.data(), n * sizeof(int));
  std::memcpy(buf.data() + n * sizeof(int), t.count.data(), n * sizeof(int));
  std::memcpy(buf.data() + 2 * n * sizeof(int), t.offset.data(), n * sizeof(int));
  std::memcpy(buf.data() + 3 * n * sizeof(int), t.w.data(), nw * sizeof(float));
  char* d = static_cast<char*>(c.staging_buffer(slot, buf.size()));
  SPLAT_HIP(hipMemcpyAsync(d, buf.data(), buf.size(), hipMemcpyHostToDevice, c.stream));
  SPLAT_HIP(hipStreamSynchronize(c.stream));  // `buf` is released on return
  ResizeTaps r;
  r.first = reinterpret_cast<const int*>(d);
  r.count = reinterpret_cast<const int*>(d + n * sizeof(int));
  r.offset = reinterpret_cast<const int*>(d + 2 * n * sizeof(int));
  r.w = reinterpret_cast<const float*>(d + 3 * n * sizeof(int));
  return r;
}

}  // namespace

void resize_device(Context& c, const uint8_t* src, int w, int h, uint8_t* dst, int nw, int nh, int filter) {
  SPLAT_CHECK(filter >= SPLAT_FILTER_TRIANGLE && filter <= SPLAT_FILTER_LANCZOS3, BAD_ARGUMENT, "resize filter");
  SPLAT_CHECK(w > 0 && h > 0 && nw > 0 && nh > 0, BAD_ARGUMENT, "resize sizes");
  if (w == nw && h == nh) {  // sample.rs resize: a copy at the same size
    SPLAT_HIP(hipMemcpyAsync(dst, src, size_t(w) * h * 4, hipMemcpyDeviceToDevice, c.stream));
    return;
  }
  const ResizeTaps rows = upload_taps(c, SLOT_ROWS, resize_taps(h, nh, filter));
  const ResizeTaps cols = upload_taps(c, SLOT_COLS, resize_taps(w, nw, filter));
  float* tmp = static_cast<float*>(c.staging_buffer(SLOT_TMP, size_t(nh) * w * 4 * sizeof(float)));
  resize_rgba8(c.ex, src, w, h, tmp, dst, nw, nh, rows, cols);
  SPLAT_HIP(hipStreamSynchronize(c.stream));  // the taps' staging is reused by the next resize
}

namespace {

void crop_into(Context& c, const uint8_t* src, int w, int left, int top, int cw, int ch, uint8_t* dst) {
  SPLAT_HIP(hipMemcpy2DAsync(dst, size_t(cw) * 4, src + (size_t(top) * w + left) * 4, size_t(w) * 4, size_t(cw) * 4,
                             size_t(ch), hipMemcpyDeviceToDevice, c.stream));
}

// One image of a batch: host pixels, the resize steps (width, height, filter; a step to the current
// size is none) and the crop of the last result.
struct Photo {
  const uint8_t* host;
  int w, h;
  std::vector<std::array<int, 3>> steps;
  int left, top;
};

// CPUs that this process may run on.
int usable_cpus() {
  cpu_set_t set;
  return sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : int(std::thread::hardware_concurrency());
}

// Memory that the GPU cannot read by itself (not page-locked, managed or device memory).
bool pageable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// Resizes and crops every photo into `batch` [n, ch, cw, 4]. The resize weights of all of them are
// computed once per (size, filter) and uploaded together; the pixels go up on the second stream into one of
// two device buffers while the previous photo is resized, pageable ones through the pinned ring,
// page-locked ones as they lie. The caller synchronises c.stream, and the host pixels have been read then.
// Six 12 MB photos: 4.0 -> 2.1 ms (uploads of pageable memory one after the other at 26 GB/s, weights
// computed for every photo, a synchronisation after each step).
void resize_batch(Context& c, const std::vector<Photo>& photos, int cw, int ch, uint8_t* batch) {
  size_t src_bytes = 0, out_bytes = 0, tmp_bytes = 0, total = 0;
  for (const Photo& p : photos) {
    SPLAT_CHECK(p.w > 0 && p.h > 0, BAD_ARGUMENT, "image size");
    int w = p.w, h = p.h;
    src_bytes = std::max(src_bytes, size_t(w) * h * 4);
    total += size_t(w) * h * 4;
    for (const auto& s : p.steps) {
      if (s[0] == w && s[1] == h) continue;
      SPLAT_CHECK(s[0] > 0 && s[1] > 0, BAD_ARGUMENT, "resize sizes");
      tmp_bytes = std::max(tmp_bytes, size_t(s[1]) * w * 4 * sizeof(float));
      out_bytes = std::max(out_bytes, size_t(s[0]) * s[1] * 4);
      w = s[0];
      h = s[1];
    }
  }
  // every buffer at its final size before anything is enqueued
  uint8_t* src[2];
  for (int k = 0; k < 2; ++k)
    src[k] = static_cast<uint8_t*>(c.staging_buffer(k ? SLOT_SRC2 : SLOT_SRC, photos.size() > size_t(k) ? src_bytes : 4));
  uint8_t* mid[2];
  for (int k = 0; k < 2; ++k) mid[k] = static_cast<uint8_t*>(c.staging_buffer(k ? SLOT_B : SLOT_A, std::max<size_t>(out_bytes, 4)));
  float* tmp = static_cast<float*>(c.staging_buffer(SLOT_TMP, std::max<size_t>(tmp_bytes, 4)));

  struct Axis { size_t at; int n; };
  std::map<std::array<int, 3>, Axis> axes;  // (in, out, filter) -> bytes into the taps
  const char* dtaps = nullptr;
  auto make_taps = [&] {
    std::vector<char> taps;
    auto axis = [&](int in, int out, int filter) {
      if (axes.count({in, out, filter})) return;
      const ResizeTapsHost t = resize_taps(in, out, filter);
      const size_t n = t.first.size(), nw = t.w.size(), at = taps.size();
      taps.resize(at + 3 * n * sizeof(int) + nw * sizeof(float));
      char* d = taps.data() + at;
      std::memcpy(d, t.first.data(), n * sizeof(int));
      std::memcpy(d + n * sizeof(int), t.count.data(), n * sizeof(int));
      std::memcpy(d + 2 * n * sizeof(int), t.offset.data(), n * sizeof(int));
      std::memcpy(d + 3 * n * sizeof(int), t.w.data(), nw * sizeof(float));
      axes[{in, out, filter}] = {at, int(n)};
    };
    for (const Photo& p : photos) {
      int w = p.w, h = p.h;
      for (const auto& s : p.steps) {
        if (s[0] == w && s[1] == h) continue;
        axis(h, s[1], s[2]);
        axis(w, s[0], s[2]);
        w = s[0];
        h = s[1];
      }
    }
    if (taps.empty()) return;
    char* d = static_cast<char*>(c.staging_buffer(SLOT_ROWS, taps.size()));
    SPLAT_HIP(hipMemcpyAsync(d, taps.data(), taps.size(), hipMemcpyHostToDevice, c.stream));
    SPLAT_HIP(hipStreamSynchronize(c.stream));  // `taps` is released on return
    dtaps = d;
  };
  auto device_taps = [&](int in, int out, int filter) {
    const Axis& a = axes.at({in, out, filter});
    ResizeTaps r;
    r.first = reinterpret_cast<const int*>(dtaps + a.at);
    r.count = r.first + a.n;
    r.offset = r.count + a.n;
    r.w = reinterpret_cast<const float*>(r.offset + a.n);
    return r;
  };
  auto process = [&](size_t k) {
    const Photo& p = photos[k];
    const uint8_t* cur = src[k & 1];
    int w = p.w, h = p.h, m = 0;
    for (const auto& s : p.steps) {
      if (s[0] == w && s[1] == h) continue;  // no resampling at the same size
      resize_rgba8(c.ex, cur, w, h, tmp, mid[m], s[0], s[1], device_taps(h, s[1], s[2]), device_taps(w, s[0], s[2]));
      cur = mid[m];
      m ^= 1;
      w = s[0];
      h = s[1];
    }
    crop_into(c, cur, w, p.left, p.top, cw, ch, batch + k * size_t(cw) * ch * 4);
  };
  std::vector<bool> direct;
  size_t staged = 0;  // bytes for the ring
  for (const Photo& p : photos) {
    direct.push_back(!pageable(p.host));
    if (!direct.back()) staged += size_t(p.w) * p.h * 4;
  }
  // A few small photos, where the ring's threads cost more than they save; or a single CPU, whose one
  // thread the driver's own staging serves as well (one 12 MB photo 580 us, through the ring 670).
  if (total < (size_t(2) << 20) || (staged > 0 && usable_cpus() < 2)) {
    make_taps();
    for (size_t k = 0; k < photos.size(); ++k) {
      SPLAT_HIP(hipMemcpyAsync(src[k & 1], photos[k].host, size_t(photos[k].w) * photos[k].h * 4, hipMemcpyHostToDevice, c.stream));
      process(k);
    }
    return;
  }
  HostRing& ring = c.host_ring();
  std::vector<RingFill::Chunk> chunks;
  for (size_t k = 0; k < photos.size(); ++k) {
    const size_t bytes = size_t(photos[k].w) * photos[k].h * 4;
    for (size_t o = 0; !direct[k] && o < bytes; o += RingFill::CHUNK)
      chunks.push_back({photos[k].host + o, std::min(RingFill::CHUNK, bytes - o)});
  }
  // the copies start after what c.stream holds (an earlier call's readers of `src`)
  SPLAT_HIP(hipEventRecord(ring.used[0], c.stream));
  SPLAT_HIP(hipStreamWaitEvent(c.aux, ring.used[0], 0));
  RingFill fill(ring.base, std::move(chunks));
  struct Drain {  // the ring is free again on return, also when an error leaves early
    Context& c;
    ~Drain() { (void)hipStreamSynchronize(c.aux); }
  } drain{c};
  size_t i = 0, landed = 0;  // chunks handed to the GPU, and those known to have arrived
  auto hand_over = [&](size_t k) {
    if (k >= 2) SPLAT_HIP(hipStreamWaitEvent(c.aux, ring.used[k & 1], 0));  // photo k - 2 has been read
    const size_t bytes = size_t(photos[k].w) * photos[k].h * 4;
    if (direct[k]) SPLAT_HIP(hipMemcpyAsync(src[k & 1], photos[k].host, bytes, hipMemcpyHostToDevice, c.aux));
    for (size_t at = 0; !direct[k] && at < bytes; at += fill.bytes(i++)) {
      while (!fill.filled(i)) {
        if (fill.help()) continue;
        if (landed < i) {
          hipError_t e = hipEventQuery(ring.sent[landed % RingFill::SLOTS]);
          if (e == hipErrorNotReady) {
            (void)hipGetLastError();  // no error: the launches below ask for theirs
            // the ring is full: nothing moves before this copy has ended
            if (!fill.has_room(i)) e = hipEventSynchronize(ring.sent[landed % RingFill::SLOTS]);
          }
          if (e != hipErrorNotReady) {
            SPLAT_HIP(e);
            ++landed;
            fill.free_one();
            continue;
          }
        }
        std::this_thread::yield();  // a worker is copying the chunk, 2 MB
      }
      const size_t slot = i % RingFill::SLOTS;
      SPLAT_HIP(hipMemcpyAsync(src[k & 1] + at, ring.base + slot * RingFill::CHUNK, fill.bytes(i), hipMemcpyHostToDevice, c.aux));
      SPLAT_HIP(hipEventRecord(ring.sent[slot], c.aux));
    }
    SPLAT_HIP(hipEventRecord(ring.copied[k & 1], c.aux));
  };
  // Photo k goes up while photo k - 1 is resized; the weights are computed under the first two's copies.
  const size_t n = photos.size();
  for (size_t k = 0; k <= n; ++k) {
    if (k < n) hand_over(k);
    if (k == std::min<size_t>(1, n - 1)) make_taps();
    if (k == 0) continue;
    SPLAT_HIP(hipStreamWaitEvent(c.stream, ring.copied[(k - 1) & 1], 0));
    process(k - 1);
    SPLAT_HIP(hipEventRecord(ring.used[(k - 1) & 1], c.stream));
  }
}

}  // namespace

void model_input(Context& c, const uint8_t* rgba, int V, int H, int W, float* images, uint8_t* foreground) {
  int* flags = static_cast<int*>(c.staging_buffer(SLOT_FLAGS, size_t(V) * sizeof(int)));
  to_model_input(c.ex, rgba, V, H, W, images, foreground);
  foreground_any(c.ex, rgba, V, H, W, flags);
  std::vector<int> any(V);
  SPLAT_HIP(hipMemcpyAsync(any.data(), flags, size_t(V) * sizeof(int), hipMemcpyDeviceToHost, c.stream));
  SPLAT_HIP(hipStreamSynchronize(c.stream));
  for (int v = 0; v < V; ++v)  // image_input.rs:197 ensure!
    SPLAT_CHECK(any[v] != 0, BAD_ARGUMENT, "view " + std::to_string(v) + " is fully transparent after cropping");
}

void da3_model_inputs(Context& c, int n, const uint8_t* const* rgba, const int* widths, const int* heights, float* images,
                      uint8_t* foreground, int& H, int& W) {
  SPLAT_CHECK(n > 0 && rgba && widths && heights && images, BAD_ARGUMENT, "model_inputs args");
  std::vector<std::array<int, 4>> sz(n);
  int cw = 1 << 30, ch = 1 << 30;
  for (int k = 0; k < n; ++k) {
    SPLAT_CHECK(rgba[k] != nullptr, BAD_ARGUMENT, "model_inputs: missing image");
    da3_model_input_size(widths[k], heights[k], sz[k][0], sz[k][1], sz[k][2], sz[k][3]);
    cw = std::min(cw, sz[k][2]);
    ch = std::min(ch, sz[k][3]);
  }
  uint8_t* batch = static_cast<uint8_t*>(c.staging_buffer(SLOT_BATCH, size_t(n) * cw * ch * 4));
  std::vector<Photo> photos;
  for (int k = 0; k < n; ++k) {
    // preprocess.rs:59-64 resize_for_model: to the bounded size, then to the patch multiples;
    // preprocess.rs:67-72 center_crop to the common size
    const int w = widths[k], h = heights[k];
    photos.push_back({rgba[k], w, h,
                      {{sz[k][0], sz[k][1], da3_resize_filter(w, h, sz[k][0], sz[k][1])},
                       {sz[k][2], sz[k][3], da3_resize_filter(sz[k][0], sz[k][1], sz[k][2], sz[k][3])}},
                      (sz[k][2] - cw) / 2, (sz[k][3] - ch) / 2});
  }
  resize_batch(c, photos, cw, ch, batch);
  model_input(c, batch, n, ch, cw, images, foreground);
  H = ch;
  W = cw;
}

void ma_model_inputs(Context& c, int n, const uint8_t* const* rgba, const int* widths, const int* heights, float* images,
                     uint8_t* foreground, int& H, int& W) {
  SPLAT_CHECK(n > 0 && rgba && widths && heights && images, BAD_ARGUMENT, "model_inputs args");
  int tw, th;
  ma_input_size(n, widths, heights, tw, th);
  uint8_t* batch = static_cast<uint8_t*>(c.staging_buffer(SLOT_BATCH, size_t(n) * tw * th * 4));
  std::vector<Photo> photos;
  for (int k = 0; k < n; ++k) {
    SPLAT_CHECK(rgba[k] != nullptr, BAD_ARGUMENT, "model_inputs: missing image");
    int rw, rh, left, top, filter;
    ma_cover(widths[k], heights[k], tw, th, rw, rh, left, top, filter);
    photos.push_back({rgba[k], widths[k], heights[k], {{rw, rh, filter}}, left, top});
  }
  resize_batch(c, photos, tw, th, batch);
  model_input(c, batch, n, th, tw, images, foreground);
  H = th;
  W = tw;
}

}  // namespace splat
