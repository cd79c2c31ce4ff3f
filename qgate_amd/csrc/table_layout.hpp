// Host tables for one call's kernels, laid out one after another (each 256-byte aligned).
#pragma once

#include <cstring>
#include <vector>

#include "qg_runtime.hpp"

namespace qg {

// They go up in one copy from the pinned table buffer (one copy per table from pageable memory took
// about 10 us of host time each); a set that does not fit there is copied table by table. The
// caller synchronises the stream before the tables go away, and so before the next upload.
class TableLayout {
  public:
    template <class T>
    size_t add(const std::vector<T> &v) {
        const size_t at = (bytes_ + 255) & ~size_t(255);
        bytes_ = at + sizeof(T) * v.size();
        parts_.push_back(Part{at, sizeof(T) * v.size(), v.data()});
        return at;
    }
    size_t bytes() const { return bytes_; }
    void upload(char *dst) const {
        if (bytes_ == 0) return;
        if (bytes_ <= kTableBytes) {
            char *h = table_buffer();
            for (const Part &p : parts_)
                if (p.bytes > 0) std::memcpy(h + p.at, p.src, p.bytes);
            QG_HIP(hipMemcpyAsync(dst, h, bytes_, hipMemcpyHostToDevice, stream()));
            return;
        }
        for (const Part &p : parts_)
            if (p.bytes > 0) QG_HIP(hipMemcpyAsync(dst + p.at, p.src, p.bytes, hipMemcpyHostToDevice, stream()));
    }

  private:
    struct Part {
        size_t at, bytes;
        const void *src;
    };
    std::vector<Part> parts_;
    size_t bytes_ = 0;
};

}  // namespace qg
