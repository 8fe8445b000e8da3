// Idle blocks of one device by size class and age (host data only; the pool in
// ngpb_api.hip owns the memory and the lock).
#pragma once
#include <cstddef>
#include <list>
#include <map>
#include <vector>

namespace ngpb {

class IdleBlocks {
 public:
  size_t bytes() const { return bytes_; }

  void put(void* p, size_t size) {
    by_size_.emplace(size, blocks_.insert(blocks_.end(), Block{size, p}));
    bytes_ += size;
  }

  // a block of exactly this size class, nullptr if there is none
  void* take(size_t size) {
    auto f = by_size_.find(size);
    if (f == by_size_.end()) return nullptr;
    void* p = f->second->p;
    blocks_.erase(f->second);
    by_size_.erase(f);
    bytes_ -= size;
    return p;
  }

  // moves the oldest blocks to `out` until at most `keep` bytes stay: blocks that nobody
  // takes any more (sizes of meshes that are gone) leave first
  void trim(size_t keep, std::vector<void*>& out) {
    while (bytes_ > keep) {
      auto b = blocks_.begin();
      auto f = by_size_.lower_bound(b->size);
      while (f->second != b) ++f;
      by_size_.erase(f);
      bytes_ -= b->size;
      out.push_back(b->p);
      blocks_.erase(b);
    }
  }

 private:
  struct Block {
    size_t size;
    void* p;
  };
  std::list<Block> blocks_;  // oldest first
  std::multimap<size_t, std::list<Block>::iterator> by_size_;
  size_t bytes_ = 0;
};

}  // namespace ngpb
