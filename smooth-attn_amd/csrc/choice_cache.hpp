// Choices of the last 16 shapes asked for, for host estimates that cost up to
// ~0.1 ms: a program asks for the same shapes again.
#pragma once

#include <algorithm>
#include <mutex>

namespace sa {

class ChoiceCache {
  public:
    template <typename Compute>
    int get(const int (&key)[6], Compute compute) {
        {
            std::lock_guard<std::mutex> lock(mu_);
            for (int i = 0; i < n_cached_; ++i)
                if (std::equal(key, key + 6, cache_[i].key)) return cache_[i].choice;
        }
        const int n = compute();
        std::lock_guard<std::mutex> lock(mu_);
        Entry& e = cache_[next_];
        std::copy(key, key + 6, e.key);
        e.choice = n;
        next_ = (next_ + 1) % kEntries;
        n_cached_ = std::min(n_cached_ + 1, kEntries);
        return n;
    }

  private:
    static constexpr int kEntries = 16;
    struct Entry {
        int key[6];
        int choice;
    };
    std::mutex mu_;
    Entry cache_[kEntries];
    int n_cached_ = 0, next_ = 0;
};

}  // namespace sa
