// build_expansion (csrc/expand.cpp) when memory runs out: the k-th allocation
// of the build, in whichever thread makes it, fails, for k spread over the whole
// build. Every build must report it as std::bad_alloc, and one without a failure
// succeed. Prints "ok" and the number of builds that failed; a build that ends
// the process shows as that.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <fstream>
#include <iterator>
#include <new>

#include "../../dpa4c-scale-aware-md_amd/csrc/expand.h"
#include "../../dpa4c-scale-aware-md_amd/csrc/model.h"

static std::atomic<long> left{-1};  // allocations until one fails; < 0: none does
static std::atomic<long> made{0};

void* operator new(std::size_t n) {
  ++made;
  if (left.load() >= 0 && left.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

using namespace dpamd;
namespace dpamd {
bool emb_supported(int, int, int) { return true; }
}  // namespace dpamd

int main(int, char** argv) {
  std::ifstream in(argv[1], std::ios::binary);
  const std::vector<unsigned char> buf((std::istreambuf_iterator<char>(in)), {});
  ModelHost m;
  if (!parse_model(buf.data(), buf.size(), m).empty()) return 1;
  made = 0;
  ExpandHost whole;
  if (!build_expansion(m, whole)) return 2;
  const long total = made;
  int failed = 0;
  for (long k = 0; k < total; k += k < 64 ? 1 : 1 + k / 16) {
    ExpandHost e;
    left = k;
    try {
      // (a failure while a thread is made only leaves fewer threads)
      if (!build_expansion(m, e) || e.fwd != whole.fwd) return 3;
    } catch (const std::bad_alloc&) {
      ++failed;
    }
    left = -1;
  }
  std::printf("ok %d\n", failed);
  return 0;
}
