// Names and short lists that a launch puts together: nothing here allocates below its fixed room.  (With std::string and std::vector a launch
// allocated 8 to 15 times and spent 1.1 us in this library on top of the runtime's 2.5.)
#pragma once
#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <string_view>
#include <vector>

namespace cutile {

// A kernel's or a shape class's name.  Longer text than its room is cut off, and is then the name of nothing.
class Name {
  uint8_t n_ = 0;
  char s_[47];   // (the longest name of a kernel has 34)

 public:
  Name() { s_[0] = 0; }
  Name(const char* t) : Name(std::string_view(t)) {}
  Name(const std::string& t) : Name(std::string_view(t)) {}
  Name(std::string_view t) { s_[0] = 0, *this += t; }
  const char* c_str() const { return s_; }
  size_t size() const { return n_; }
  bool empty() const { return n_ == 0; }
  void clear() { s_[n_ = 0] = 0; }
  operator std::string_view() const { return {s_, n_}; }
  Name& operator+=(std::string_view t) {
    const size_t n = std::min(t.size(), sizeof(s_) - 1 - n_);
    memcpy(s_ + n_, t.data(), n);
    s_[n_ += (uint8_t)n] = 0;
    return *this;
  }
  Name& operator+=(const char* t) { return *this += std::string_view(t); }
};
inline bool operator==(const Name& a, const Name& b) { return a.size() == b.size() && memcmp(a.c_str(), b.c_str(), a.size()) == 0; }
inline bool operator==(const Name& a, const char* b) { return strcmp(a.c_str(), b) == 0; }
inline bool operator!=(const Name& a, const Name& b) { return !(a == b); }
inline bool operator!=(const Name& a, const char* b) { return !(a == b); }
inline Name operator+(Name a, const Name& b) { return a += std::string_view(b); }
inline Name operator+(Name a, const char* b) { return a += b; }
inline Name operator+(const char* a, const Name& b) { return Name(a) += std::string_view(b); }

// A whole number as text.
inline Name num(int64_t v) {
  char text[24], *end = text + sizeof(text), *p = end;
  uint64_t u = v < 0 ? 0 - (uint64_t)v : (uint64_t)v;
  do *--p = (char)('0' + u % 10);
  while (u /= 10);
  if (v < 0) *--p = '-';
  return Name(std::string_view(p, (size_t)(end - p)));
}

// A list whose first N items need no allocation.
template <typename T, size_t N>
class Few {
  size_t n_ = 0;
  T few_[N];
  std::vector<T> many_;   // all of them, once there are more than N

 public:
  Few() {}
  Few(std::initializer_list<T> items) {
    for (const T& t : items) push_back(t);
  }
  void push_back(const T& t) {
    if (n_ < N) {
      few_[n_] = t;
    } else {
      if (many_.empty()) many_.assign(few_, few_ + N);
      many_.push_back(t);
    }
    ++n_;
  }
  size_t size() const { return n_; }
  bool empty() const { return n_ == 0; }
  T* begin() { return many_.empty() ? few_ : many_.data(); }
  T* end() { return begin() + n_; }
  const T* begin() const { return many_.empty() ? few_ : many_.data(); }
  const T* end() const { return begin() + n_; }
  const T& operator[](size_t i) const { return begin()[i]; }
};
using Names = Few<Name, 6>;

// Sorts a short list in place; equal items keep their order.
template <typename It, typename Less>
void sort_few(It first, It last, Less less) {
  for (It i = first; i != last; ++i)
    for (It j = i; j != first && less(*j, *(j - 1)); --j) std::swap(*j, *(j - 1));
}

}  // namespace cutile
