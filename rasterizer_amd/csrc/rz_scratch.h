// Working memory of a context's scene preparation (rz_sah_batches,
// rz_quad_decompose_device, rz_bake_device, rz_prepare_*), kept between calls:
// allocating and freeing a buffer of some megabytes takes about 0.3 ms, more
// than most of the kernels that use it.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace rzd {

// Device memory handed out in 256-byte aligned parts, released in the reverse
// order (Frame).  A call that needs more than is there gets further blocks; after
// it they are given back and the next call allocates one block of half as much
// again as was in use, for calls that grow.  More than kKeepDevice is not kept,
// and the next call allocates so much at once only when its first part or block is
// a fair share of it.
// Used by one context's calls, on its stream, by one thread at a time, so a
// part is only handed on to work that the stream orders behind its last use;
// everything is freed with the context.
class Scratch {
 public:
  static constexpr size_t kKeepDevice = size_t(256) << 20;
  static constexpr size_t kMaxHost = size_t(64) << 20;

  ~Scratch() {
    free_blocks();
    if (host_) (void)hipHostFree(host_);
  }

  // Device memory until the enclosing Frame ends; null when there is none.
  template <typename T>
  T* take(size_t count) {
    size_t bytes = (count * sizeof(T) + 255) & ~size_t(255);
    if (bytes == 0) bytes = 256;
    while (cur_ < nBlocks_ && used_ + bytes > blocks_[cur_].size) {
      before_ += blocks_[cur_++].size;
      used_ = 0;
    }
    if (cur_ == nBlocks_) {
      if (nBlocks_ == kMaxBlocks) return nullptr;
      Block b;
      const bool alike = want_ <= kKeepDevice ? nBlocks_ == 0 : before_ + bytes >= want_ / 16;
      const size_t more = alike && before_ < want_ ? want_ - before_ : 0;
      if (more > bytes && hipMalloc(&b.base, more) == hipSuccess) {
        b.size = more;
      } else {
        (void)hipGetLastError();
        if (hipMalloc(&b.base, bytes) != hipSuccess) {
          (void)hipGetLastError();
          return nullptr;
        }
        b.size = bytes;
      }
      blocks_[nBlocks_++] = b;
      used_ = 0;
    }
    T* p = reinterpret_cast<T*>(static_cast<unsigned char*>(blocks_[cur_].base) + used_);
    used_ += bytes;
    live_ += bytes;
    peak_ = peak_ > live_ ? peak_ : live_;
    return p;
  }

  // Pinned host memory (one user at a time), or null when it cannot be had or
  // would exceed kMaxHost.
  void* host(size_t bytes) {
    if (bytes > kMaxHost) return nullptr;
    if (bytes > hostBytes_) {
      const size_t twice = 2 * hostBytes_ < kMaxHost ? 2 * hostBytes_ : kMaxHost;  // pinning is slow: grow seldom
      if (host_) (void)hipHostFree(host_);
      host_ = nullptr;
      hostBytes_ = 0;
      const size_t size = bytes > twice ? bytes : twice;
      if (hipHostMalloc(&host_, size) != hipSuccess) {
        (void)hipGetLastError();
        host_ = nullptr;
        return nullptr;
      }
      hostBytes_ = size;
    }
    return host_;
  }

  // Parts taken while a Frame lives are released when it ends.
  class Frame {
   public:
    explicit Frame(Scratch& s) : s_(s), cur_(s.cur_), used_(s.used_), before_(s.before_), live_(s.live_) { ++s_.depth_; }
    ~Frame() {
      s_.cur_ = cur_;
      s_.used_ = used_;
      s_.before_ = before_;
      s_.live_ = live_;
      if (--s_.depth_ == 0) s_.trim();
    }
    Frame(const Frame&) = delete;
    Frame& operator=(const Frame&) = delete;

   private:
    Scratch& s_;
    size_t cur_, used_, before_, live_;
  };

 private:
  struct Block {
    void* base = nullptr;
    size_t size = 0;
  };

  void free_blocks() {
    for (size_t i = 0; i < nBlocks_; ++i) (void)hipFree(blocks_[i].base);  // waits for the work that uses it
    nBlocks_ = cur_ = used_ = before_ = live_ = 0;
  }
  void trim() {
    const size_t more = peak_ + peak_ / 2;
    want_ = peak_ > kKeepDevice ? peak_ : more < kKeepDevice ? more : kKeepDevice;
    if (nBlocks_ > 1 || (nBlocks_ == 1 && blocks_[0].size > kKeepDevice)) free_blocks();
    peak_ = 0;
  }

  // A call takes at most 46 parts (rz_prepare_mesh_device: 2 of its own, 11 of
  // the decomposition, 4 of the scene, 24 of the SAH pass, 5 of the bake).
  static constexpr size_t kMaxBlocks = 64;
  Block blocks_[kMaxBlocks];
  size_t nBlocks_ = 0;
  size_t cur_ = 0, used_ = 0;  // the next part starts at blocks_[cur_].base + used_
  size_t before_ = 0;          // the sizes of the blocks before it
  size_t live_ = 0;            // the parts handed out: one block would hold as much
  size_t peak_ = 0, want_ = 0;
  int depth_ = 0;
  void* host_ = nullptr;
  size_t hostBytes_ = 0;
};

}  // namespace rzd
