// Reading a handle's solution vectors one after the other (host code; also compiled
// by a plain C++ compiler for the CPU checks).
//
// A copy with its own synchronisation costs 11-17 us however short it is, so the
// second call in a row fetches the next few vectors in one launch and the window
// doubles while the calls stay in order, to READ_ROWS vectors or READ_BYTES.  A first
// or a random access fetches its own vector alone.  Measured on MI355X, 512 signals
// of 16384 with their 4096 measurements: 42 us a signal one by one, 14 us in order.
//
// The window holds what the device memory holds: whatever can write the handle's
// vectors does so under a ReadAhead::Writing, which drops the window before and
// after, since a read from another thread may open one in between.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>

constexpr int READ_ROWS = 64;
constexpr size_t READ_BYTES = (size_t)4 << 20;
class ReadAhead {
 public:
  // How the window's memory is made and given back (null: no memory).
  ReadAhead(float *(*alloc)(size_t), void (*release)(float *)) : alloc_(alloc), release_(release) {}
  ReadAhead(const ReadAhead &) = delete;
  ~ReadAhead() {
    if (buf_) release_(buf_);
  }
  class Writing {
   public:
    explicit Writing(ReadAhead &r) : r_(r) { r_.drop(); }
    ~Writing() { r_.drop(); }
    Writing(const Writing &) = delete;

   private:
    ReadAhead &r_;
  };
  // Row i of `count`: piece(i, p, &src, &n) gives its p-th piece (one or two of
  // them), out[p] takes it where not null; a window is fetched by add(src, dst, n) for
  // each piece, then run().  False: the caller copies by itself (no window for this
  // call, or no memory).
  template <class F, class Add, class Run>
  bool get(int i, int count, int pieces, F piece, float *const out[2], Add add, Run run) {
    std::lock_guard<std::mutex> lock(mu_);
    if (i < first_ || i >= first_ + cnt_) {
      win_ = i == next_ ? std::min(READ_ROWS, std::max(4, 2 * win_)) : 0;
      next_ = i + 1;
      cnt_ = 0;
      if (!win_) return false;
      size_t used = 0;
      const int top = std::min(win_, count - i);
      const float *src[2];
      long n[2];
      int w = 0;
      for (; w < top; w++) {
        size_t row = 0;
        for (int p = 0; p < pieces; p++) {
          piece(i + w, p, &src[p], &n[p]);
          row += ((size_t)n[p] + 15) / 16 * 16;
        }
        if (4 * (used + row) > READ_BYTES) break;
        if (!buf_ && !(buf_ = alloc_(READ_BYTES))) return false;
        for (int p = 0; p < pieces; p++) {
          off_[w][p] = used;
          add(src[p], buf_ + used, n[p]);
          used += ((size_t)n[p] + 15) / 16 * 16;
        }
      }
      if (!w || !run()) return false;
      first_ = i;
      cnt_ = w;
    }
    next_ = i + 1;
    for (int p = 0; p < pieces; p++) {
      const float *src;
      long n;
      piece(i, p, &src, &n);
      if (out[p]) memcpy(out[p], buf_ + off_[i - first_][p], sizeof(float) * (size_t)n);
    }
    return true;
  }

 private:
  void drop() {
    std::lock_guard<std::mutex> lock(mu_);
    cnt_ = win_ = 0;
    next_ = -1;
  }
  float *(*alloc_)(size_t);
  void (*release_)(float *);
  std::mutex mu_;
  float *buf_ = nullptr;
  int first_ = 0, cnt_ = 0, next_ = -1, win_ = 0;
  size_t off_[READ_ROWS][2];
};
