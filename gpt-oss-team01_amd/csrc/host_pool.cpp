// Memory of results in host arrays, kept for the next result of its size where the array it was last used for is gone: the
// first touch of fresh pages costs ten times the copy into them (3 MB of logits: 700 us of page faults, 40 us of copying).
// Arrays get it through numpy's memory handlers, so they own it like any other array's (resize in place included), and it
// comes back with the last array or view over it.  At most `limit` bytes are kept; what was returned longest ago goes
// first, so sizes that are no longer asked for do not stay in the way.  No entry throws or allocates but by malloc.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <mutex>
#include <new>

namespace {

// What numpy's C API reads through a capsule named "mem_handler" (PyDataMem_Handler, version 1).
struct Handler {
  char name[127];
  uint8_t version;
  void *pool;
  void *(*malloc)(void *, size_t);
  void *(*calloc)(void *, size_t, size_t);
  void *(*realloc)(void *, void *, size_t);
  void (*free)(void *, void *, size_t);
};

// In front of every block's memory.  The size numpy passes to free is the array's at that time, which need not be this.
struct alignas(64) Block {
  size_t bytes;
  Block *older, *newer;   // while kept
};

constexpr size_t PAGE = 4096;
constexpr int LOOK = 256;   // kept blocks that a request looks at, the last returned first

struct Pool {
  Handler handler;
  std::mutex mu;
  size_t limit, kept = 0, used = 0;   // bytes kept; blocks in use, and one while the owner has not released the pool
  Block *oldest = nullptr, *newest = nullptr;

  void unlink(Block *b) {
    (b->older ? b->older->newer : oldest) = b->newer;
    (b->newer ? b->newer->older : newest) = b->older;
    kept -= b->bytes;
  }
  void drop(size_t most) {
    while (kept > most) {
      Block *b = oldest;
      unlink(b);
      ::free(b);
    }
  }
};

Block *block_of(void *memory) { return reinterpret_cast<Block *>(memory) - 1; }

void *take(void *ctx, size_t n) {
  Pool *p = static_cast<Pool *>(ctx);
  if (n > SIZE_MAX - 2 * PAGE) return nullptr;
  const size_t bytes = (n + PAGE - 1) / PAGE * PAGE;
  Block *found = nullptr;
  {
    std::lock_guard<std::mutex> lock(p->mu);
    int left = LOOK;
    for (Block *b = p->newest; b && left > 0 && !found; b = b->older, left--)
      if (b->bytes == bytes) found = b;
    if (found) {
      p->unlink(found);
      p->used++;
      return found + 1;
    }
  }
  Block *b = static_cast<Block *>(aligned_alloc(alignof(Block), sizeof(Block) + bytes));
  if (!b) return nullptr;
  b->bytes = bytes;
  std::lock_guard<std::mutex> lock(p->mu);
  p->used++;
  return b + 1;
}

// one user less; the pool's own memory goes with the last
void leave(Pool *p, Block *b) {
  bool last;
  {
    std::lock_guard<std::mutex> lock(p->mu);
    if (b && b->bytes <= p->limit) {
      p->drop(p->limit - b->bytes);
      b->older = p->newest;
      b->newer = nullptr;
      (p->newest ? p->newest->newer : p->oldest) = b;
      p->newest = b;
      p->kept += b->bytes;
      b = nullptr;
    }
    last = --p->used == 0;
  }
  ::free(b);
  if (last) {
    p->drop(0);
    delete p;
  }
}

void give(void *ctx, void *memory, size_t) {
  if (memory) leave(static_cast<Pool *>(ctx), block_of(memory));
}

void *take_zeroed(void *ctx, size_t count, size_t size) {
  if (size && count > SIZE_MAX / size) return nullptr;
  void *m = take(ctx, count * size);
  return m ? memset(m, 0, count * size) : nullptr;
}

void *take_larger(void *ctx, void *memory, size_t n) {
  if (!memory) return take(ctx, n);
  const size_t had = block_of(memory)->bytes;
  if (n <= had) return memory;
  void *m = take(ctx, n);
  if (!m) return nullptr;
  memcpy(m, memory, had);
  give(ctx, memory, had);
  return m;
}

}  // namespace

// For engine.py: a pool, whose first member is the handler; the memory it keeps now; up to n sizes of the blocks it keeps,
// the oldest first, and their number.  A released pool keeps nothing and ends with the last array over its memory.
extern "C" void *gptoss_host_pool_create(size_t limit) {
  Pool *p = new (std::nothrow) Pool;
  if (!p) return nullptr;
  p->handler = {"gptoss_results", 1, p, take, take_zeroed, take_larger, give};
  p->limit = limit;
  p->used = 1;
  return p;
}

extern "C" void gptoss_host_pool_release(void *pool) {
  Pool *p = static_cast<Pool *>(pool);
  {
    std::lock_guard<std::mutex> lock(p->mu);
    p->limit = 0;
    p->drop(0);
  }
  leave(p, nullptr);
}

extern "C" size_t gptoss_host_pool_kept(void *pool, size_t *sizes, size_t n, size_t *count) {
  Pool *p = static_cast<Pool *>(pool);
  std::lock_guard<std::mutex> lock(p->mu);
  *count = 0;
  for (Block *b = p->oldest; b; b = b->newer, ++*count)
    if (*count < n) sizes[*count] = b->bytes;
  return p->kept;
}
