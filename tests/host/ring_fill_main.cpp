// RingFill against a stand-in for the GPU: chunks that are handed over land some steps later, in order.
// argv: bytes of each image, comma separated (0 is none). Prints "ok" once every image has come through
// whole; with the first argument "abandon" it leaves after half the chunks instead.
#include <cstdio>
#include <cstdlib>
#include <deque>
#include <random>
#include <string>

#include "../../splatting-rs_amd/csrc/ring_fill.h"

using splat::RingFill;

int main(int argc, char** argv) {
  if (argc < 3) return 2;
  const bool abandon = std::string(argv[1]) == "abandon";
  std::vector<std::vector<uint8_t>> images;
  std::mt19937 rng(7);
  for (char* p = argv[2]; *p;) {
    images.emplace_back(std::strtoul(p, &p, 10));
    for (auto& b : images.back()) b = uint8_t(rng());
    if (*p == ',') ++p;
  }
  std::vector<RingFill::Chunk> chunks;
  for (const auto& im : images)
    for (size_t o = 0; o < im.size(); o += RingFill::CHUNK) chunks.push_back({im.data() + o, std::min(RingFill::CHUNK, im.size() - o)});
  const size_t n = chunks.size();
  std::vector<uint8_t> ring(RingFill::SLOTS * RingFill::CHUNK), out;
  RingFill fill(ring.data(), chunks);
  std::deque<size_t> flight;  // handed over, not landed: their slots may not change
  auto land = [&] {
    const size_t i = flight.front();
    flight.pop_front();
    const uint8_t* s = ring.data() + (i % RingFill::SLOTS) * RingFill::CHUNK;
    out.insert(out.end(), s, s + fill.bytes(i));
    fill.free_one();
  };
  for (size_t i = 0; i < n; ++i) {
    while (!fill.filled(i)) {
      if (fill.help()) continue;
      if (!flight.empty() && (!fill.has_room(i) || rng() % 4 == 0)) land();
      else std::this_thread::yield();
    }
    flight.push_back(i);
    if (abandon && i == n / 2) return std::puts("abandoned"), 0;
  }
  while (!flight.empty()) land();
  std::vector<uint8_t> want;
  for (const auto& im : images) want.insert(want.end(), im.begin(), im.end());
  return std::puts(out == want ? "ok" : "differs"), out == want ? 0 : 1;
}
