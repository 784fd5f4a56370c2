// Words of host memory through which kernels send the host numbers that it waits for.  (Nothing here needs a GPU: Runtime
// stands for the calls that do.)
#pragma once

#include <stdint.h>

#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace omni_attn {

// Where the workgroups of a kernel write a count each that the host waits for, as words of a tag and the count:
// pinned host memory, handed out per call (so calls of several threads and streams do not meet) and taken
// back; at most kKeep pieces of kWords words are kept between calls.
// Runtime: Stream; allocate(bytes), which throws, and release(memory); running(stream), which throws the stream's error;
// drain(stream): waits for everything on the stream, false where that cannot be done.
template <class Runtime, int kCountBits>
class HostCounts {
 public:
  typedef typename Runtime::Stream Stream;
  // (a word per query block costs the host 10 ns and more; their sum costs two launches more.  A call, us, with words /
  // with their sum: 512 query blocks 33 / 31, 1024 35 / 34, 2048 62 / 41, 4096 98 / 54)
  static constexpr int kWords = 512;
  static constexpr size_t kKeep = 16;
  HostCounts() {
    {
      std::lock_guard<std::mutex> lock(mutex());
      if (!spare().empty()) {
        words_ = spare().back();
        spare().pop_back();
        return;
      }
    }
    words_ = static_cast<uint32_t*>(Runtime::allocate(size_t(kWords + 16) * 4));
    std::memset(words_, 0, size_t(kWords + 16) * 4);
  }
  ~HostCounts() {
    if (pending_) {
      // The call failed with a kernel under way, or refused, that may write here: it is waited for.  (Memory of a stream
      // that cannot be waited for -- one that is captured, a device that reported an error -- stays allocated.)
      if (!Runtime::drain(stream_)) return;
      std::memset(words_, 0, size_t(kWords) * 4);
    }
    {
      std::lock_guard<std::mutex> lock(mutex());
      if (spare().size() < kKeep) {
        spare().push_back(words_);
        return;
      }
    }
    Runtime::release(words_);
  }
  HostCounts(const HostCounts&) = delete;
  HostCounts& operator=(const HostCounts&) = delete;

  uint32_t* memory() { return words_; }
  // A tag that no word has, for a kernel that is launched on `stream` next: words are cleared where the tags begin again.
  int next_tag(Stream stream) {
    uint32_t& last = words_[kWords];
    if (last == (1u << (32 - kCountBits)) - 1) {
      std::memset(words_, 0, size_t(kWords) * 4);
      last = 0;
    }
    pending_ = true;
    stream_ = stream;
    return int(++last);
  }
  // The sum of the first n counts, once the kernel that writes them has run.
  int64_t wait(int tag, int n) {
    int64_t sum = 0;
    for (int i = 0; i < n; ++i) sum += wait_for(i, tag) & ((1u << kCountBits) - 1);
    pending_ = false;
    return sum;
  }
  // A number of any size in word 0, written before the tag in word 1.
  int32_t wait_total(int tag) {
    (void)wait_for(1, tag);
    pending_ = false;
    const int32_t total = int32_t(words_[0]);
    words_[0] = words_[1] = 0;
    return total;
  }
  static int word_of(int tag) { return int(uint32_t(tag) << kCountBits); }

 private:
  // Ends as well when the stream has nothing left to run or reports an error.
  uint32_t wait_for(int i, int tag) {
    for (unsigned spins = 1;; ++spins) {
      const uint32_t x = __atomic_load_n(words_ + i, __ATOMIC_ACQUIRE);
      if (int(x >> kCountBits) == tag) return x;
      if (spins % 8192 == 0 && !Runtime::running(stream_) &&
          int(__atomic_load_n(words_ + i, __ATOMIC_ACQUIRE) >> kCountBits) != tag)
        throw std::runtime_error("omni_attn: the mask was not built: its kernel sent nothing");
    }
  }
  static std::mutex& mutex() {
    static std::mutex* m = new std::mutex;
    return *m;
  }
  static std::vector<uint32_t*>& spare() {
    static std::vector<uint32_t*>* v = new std::vector<uint32_t*>;
    return *v;
  }
  uint32_t* words_ = nullptr;  // kWords counts; the last tag
  bool pending_ = false;
  Stream stream_ = {};
};

}  // namespace omni_attn
