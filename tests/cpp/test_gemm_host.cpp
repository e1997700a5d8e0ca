// test_gemm_host.cpp — host side of the GEMMs, without a GPU: what
// gemm() refuses and accepts, and launch rules.  An accepted call gets as far as its launch,
// which fails here for want of a device (MFT_EHIP); a refused one throws
// MFT_EINVAL before.  The operands are addresses that nothing reads.
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <utility>

#include "gemm_common.h"

using namespace mft;

namespace {

float* at(uintptr_t a) { return reinterpret_cast<float*>(a); }

int status_of(int M, int N, int K, bool b_nk, int64_t lda, int64_t ldb, size_t ws_bytes, const KernelEvents* ev = nullptr) {
  Scratch ws;
  ws.ptr = at(0x40000000);
  ws.bytes = ws_bytes;
  try {
    gemm(nullptr, at(0x10000000), lda, at(0x20000000), ldb, b_nk, false, at(0x30000000), N, M, N, K, GemmEpilogue(), ws, ev);
  } catch (const Error& e) {
    printf("M=%d N=%d K=%d %s: %s\n", M, N, K, b_nk ? "NK" : "KN", e.what());
    return e.code;
  }
  return MFT_OK;
}

bool expect(bool ok, const char* what) {
  if (!ok) printf("FAILED: %s\n", what);
  return ok;
}

// Reductions too deep for one 32-bit buffer offset, whose slices are not: the
// plan splits every tile, whatever the tile count is a multiple of.
bool deep() {
  bool ok = true;
  struct Shape {
    int M, N, K;
    bool b_nk;
    int64_t lda, ldb;
    int slices;
  };
  const Shape shapes[] = {
      {1024, 4096, 262144, false, 262144, 4096, 2},  // dlogits·E of a 4096-wide model: 256 tiles of 128×128
      {768, 8192, 200000, false, 200000, 8192, 2},   // whole rounds of 64-row tiles, a round and a half of 128×128
      {1100, 4352, 262144, false, 262144, 4352, 2},  // not a multiple
      {64, 64, 8350000, true, 8350000, 8350000, 4},  // rows so long that A's and B's first 128 leave little for K
  };
  for (const Shape& s : shapes) {
    const size_t ws = (size_t)s.slices * s.M * s.N * sizeof(float);
    ok &= expect(status_of(s.M, s.N, s.K, s.b_nk, s.lda, s.ldb, ws + 256) == MFT_EHIP, "a deep reduction with room for its slices");
    ok &= expect(status_of(s.M, s.N, s.K, s.b_nk, s.lda, s.ldb, 0) == MFT_EINVAL, "a deep reduction without a workspace");
  }
  return ok;
}

// A call refused for its size leaves the caller's events as they were.
bool timing() {
  KernelEvents ev;
  ev.start = ev.stop = ev.tail_start = ev.tail_stop = reinterpret_cast<hipEvent_t>(at(0x50000000));
  bool ok = expect(status_of(64, 640, 1 << 20, false, 1 << 20, 1 << 20, 1 << 26, &ev) == MFT_EINVAL, "refused before any event is touched");
  ok &= expect(!ev.tail_used, "no reduction was timed");
  return ok;
}

// 16-byte output rows of a column-segmented launch: every segment's C and
// pitch count, not the first one's.
bool segments() {
  auto vec = [](std::initializer_list<std::pair<uintptr_t, int64_t>> segs) {
    GemmHSegmentArg a[3] = {};
    int n = 0;
    for (const auto& s : segs) {
      a[n].C = at(s.first);
      a[n++].ldc = s.second;
    }
    return segments_out_vec(a, n);
  };
  bool ok = expect(vec({{0x1000, 64}, {0x2000, 128}, {0x3010, 68}}), "aligned segments");
  ok &= expect(!vec({{0x1000, 64}, {0x2004, 64}}), "a second segment off by four bytes");
  ok &= expect(!vec({{0x1000, 64}, {0x2000, 64}, {0x3000, 65}}), "an odd pitch of the third");
  ok &= expect(!vec({{0x1008, 64}, {0x2000, 64}}), "a first segment off by eight bytes");
  return ok;
}

// Which products the 32×64 fp32 tiles take: at most a round of them, slices of
// K from 256 on, and no row statistics.
bool small() {
  for (int M : {8, 32, 100, 300})
    for (int N : {36, 256, 1068})
      for (int K : {260, 480, 1040, 2048, 3976, 65536}) {
        const XPlan p = plan_gemm_x(M, N, K, int64_t(1) << 28, size_t(64) << 20, false, false, true, K % 32 != 0);
        GemmParams g{};
        g.K = K;
        if (p.bm == 32 && !expect(gemm_x_depth(p, g) >= 256, "slices of small tiles")) return false;
      }
  auto bm = [](int M, int N, int K, bool stats = false, bool small = true) {
    return plan_gemm_x(M, N, K, int64_t(1) << 28, size_t(64) << 20, false, stats, small, K % 32 != 0).bm;
  };
  bool ok = expect(bm(512, 768, 768) == 32 && bm(16, 256, 256) == 32 && bm(1024, 512, 512) == 32 && bm(300, 300, 300) == 32,
                   "small products");
  ok &= expect(bm(256, 256, 255) == 64 && bm(8, 64, 64) == 64, "K below 256");
  ok &= expect(bm(1024, 640, 640) != 32 && bm(512, 3072, 768) != 32 && bm(1024, 4864, 896) != 32, "more than a round of tiles");
  ok &= expect(bm(128, 1024, 512, true) == 128, "row statistics");
  ok &= expect(bm(512, 768, 768, false, false) == 64 && bm(16, 256, 256, false, false) == 64, "the engine's products");
  return ok;
}

}  // namespace

int main(int argc, char** argv) {
  const char* mode = argc > 1 ? argv[1] : "";
  bool ok = false;
  if (!strcmp(mode, "deep")) ok = deep();
  if (!strcmp(mode, "timing")) ok = timing();
  if (!strcmp(mode, "segments")) ok = segments();
  if (!strcmp(mode, "small")) ok = small();
  puts(ok ? "OK" : "FAILED");
  return ok ? 0 : 1;
}
