// Growing host bytes: the part of std::vector<uint8_t> the decoders on the
// host use, in memory that may come from elsewhere (a context's pinned
// staging buffer, hh_internal.hpp) as long as that has room.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <cstring>
#include <memory>

namespace hh {

class HostBytes {
  public:
    // more(owner, bytes, cap): memory of at least `bytes` with the present
    // contents kept at its start and its size in *cap, or nullptr
    typedef uint8_t *(*More)(void *owner, size_t bytes, size_t *cap);
    HostBytes() = default;
    HostBytes(More more, void *owner) : more_(more), owner_(owner) {}
    HostBytes(const HostBytes &) = delete;
    HostBytes &operator=(const HostBytes &) = delete;

    uint8_t *data() { return p_; }
    const uint8_t *data() const { return p_; }
    size_t size() const { return n_; }
    bool owned() const { return own_ != nullptr; }  // not the owner's memory
    void clear() { n_ = 0; }
    void reserve(size_t n) {
        if (n > cap_) grow(n);
    }
    // added bytes are not set
    void resize(size_t n) {
        if (n > cap_) grow(n < 2 * cap_ ? 2 * cap_ : n);
        n_ = n;
    }
    void append(const uint8_t *b, size_t n) {
        if (n == 0) return;
        resize(n_ + n);
        std::memcpy(p_ + n_ - n, b, n);
    }
    void append(size_t n, uint8_t v) {
        if (n == 0) return;
        resize(n_ + n);
        std::memset(p_ + n_ - n, v, n);
    }

  private:
    void grow(size_t bytes) {
        if (more_ && !own_) {
            size_t cap = 0;
            if (uint8_t *q = more_(owner_, bytes, &cap)) {
                p_ = q;
                cap_ = cap;
                return;
            }
        }
        std::unique_ptr<uint8_t[]> v(new uint8_t[bytes]);
        if (n_) std::memcpy(v.get(), p_, n_);
        own_.swap(v);
        p_ = own_.get();
        cap_ = bytes;
    }
    uint8_t *p_ = nullptr;
    size_t n_ = 0, cap_ = 0;
    More more_ = nullptr;
    void *owner_ = nullptr;
    std::unique_ptr<uint8_t[]> own_;
};

// zstd::decode_all on the host (host_zstd.cpp): false on a malformed stream.
bool zstd_decode_all(const uint8_t *in, size_t len, HostBytes &out);

}  // namespace hh
