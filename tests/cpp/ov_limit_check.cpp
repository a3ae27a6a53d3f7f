// Host check of the overlaps' row chunks under a fixed partial-sum buffer: for
// every size, slab depth, slot count and cap the chunks are whole slabs, cover
// every row once, number no more than the cap, and take no more rows in turn
// over their rounds of resident workgroups than the cap's own count does.
// Prints one line per failure; exit status 1 if any.
#include <cstdio>

#include "../../derek_amd/csrc/ov_geom.hpp"

using namespace derek;

int main() {
  int bad = 0, checked = 0;
  for (int64_t npw : {1, 15, 16, 17, 255, 1503, 5003, 62669, 161214})
    for (int m : {1, 10, 64, 65, 160, 300, 600, 1200})
      for (int n : {1, 33, 64, 300, 600})
        for (bool herm : {false, true})
          for (int batch : {1, 3})
            for (int slots : {256, 512, 768})
              for (int ks : {OV_KS, BF_KS})
                for (int64_t cap : {0, 1, 2, 3, 5, 11, 23, 81, 1000, 1 << 21}) {
                  if (herm && m != n) continue;
                  const int64_t most = std::max<int64_t>({1, npw / 256, std::min<int64_t>(npw / 64, 128)});
                  OvGeom g = ov_geom(m, n, npw, herm, batch, slots, ks);
                  const OvGeom free = g;
                  ov_limit_chunks(g, cap, ks, batch, slots);
                  ++checked;
                  const int64_t c = cap < 1 ? free.nchunk : std::min<int64_t>(cap, free.nchunk);
                  const int64_t k = ov_ceil_div(ov_ceil_div(npw, c), ks) * ks;
                  auto rows = [&](int64_t chunks, int64_t kch) {
                    return ov_ceil_div(g.ntiles * batch * chunks, slots) * kch;
                  };
                  const bool ok = free.nchunk <= most && (int64_t)free.nchunk * free.kch >= npw &&
                                  (int64_t)(free.nchunk - 1) * free.kch < npw && g.kch % ks == 0 && g.nchunk <= c && (int64_t)g.nchunk * g.kch >= npw &&
                                  (int64_t)(g.nchunk - 1) * g.kch < npw &&
                                  (c == free.nchunk ? g.kch == free.kch && g.nchunk == free.nchunk
                                                    : rows(g.nchunk, g.kch) <= rows(ov_ceil_div(npw, k), k));
                  if (!ok) {
                    ++bad;
                    std::printf("FAIL %lld x %d x %d herm=%d batch=%d slots=%d ks=%d cap=%lld: %d chunks of %lld\n",
                                (long long)npw, m, n, (int)herm, batch, slots, ks, (long long)cap, g.nchunk,
                                (long long)g.kch);
                  }
                }
  std::printf("%d sizes checked, %d wrong\n", checked, bad);
  return bad ? 1 : 0;
}
