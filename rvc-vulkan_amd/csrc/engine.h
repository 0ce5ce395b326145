// Engine object behind the C ABI: one HIP device, one stream, a registry of
// device buffers keyed by opaque int64 ids, a growable packing scratch and
// the pending batch of the record/commit API.
#pragma once

#include <deque>
#include <list>
#include <memory>
#include <unordered_map>

#include "internal.h"

namespace rvc {

struct DevBuf {
  void* ptr = nullptr;
  size_t bytes = 0;
  size_t block = 0;  // bytes of the device block behind it (Engine::block_size)
};

struct BatchOp {
  int op;
  long long a, b, c;
  long long p[20];  // p0..p10 of rvc_batch_add, or the longer parameter lists of the segment records
};

struct Engine {
  int device = 0;
  hipStream_t stream = nullptr;
  std::mutex mu;
  std::unordered_map<long long, DevBuf> bufs;
  long long next_id = 1;
  std::string device_name;
  // Freed blocks, by size, for the next buffer of that size: an op-level call
  // allocates and frees a buffer per argument (2.3 us each by hipMalloc +
  // hipFree, in a call of its own; a LayerNorm of [100][192] 50 -> 40 us).  A
  // block goes back to the pool after the stream has been waited for, as it went
  // to hipFree before.
  // At most kPoolBytes are kept, the oldest given back first, blocks above
  // kPoolBlock not at all; the pool is emptied where any device allocation of
  // the engine or its sessions fails (dev_malloc), and with the engine.
  static constexpr size_t kPoolBytes = 128u << 20, kPoolBlock = 32u << 20;
  struct PoolBlock {
    void* ptr;
    size_t bytes;
  };
  std::list<PoolBlock> pool;  // oldest first
  std::unordered_map<size_t, std::deque<std::list<PoolBlock>::iterator>> pool_of;  // by size, oldest first
  size_t pool_bytes = 0;
  // Pinned staging of small transfers: an upload is copied here and on to the
  // device, by a kernel of the stream and without waiting; a download comes back
  // the same way.  (A copy engine's hand-over to and from the stream costs more
  // than the copy: the same LayerNorm 40 -> 32 us, a 192 -> 768 conv of 100 columns
  // 62 -> 52 us.)  `stage_used` starts again at every wait for the stream.
  // Transfers above kStageMax go straight from / to the caller's memory (equal at
  // 1 MB).
  static constexpr size_t kStageBytes = 4u << 20, kStageMax = 1u << 20;
  char* stage = nullptr;
  size_t stage_used = 0;
  // scratch for packed weights of op-level calls
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  // BiGRU exchange words + error flag of rvc_gru / rvc_batch_add_gru (kept
  // apart from the scratch, which later ops of a batch reuse), and whether a
  // launched GRU's flag still awaits its check after the next sync
  unsigned long long* gru_state = nullptr;
  bool gru_pending = false;
  // record/commit batch
  std::vector<BatchOp> batch;
  bool in_flight = false;
  // GPU-busy accounting behind rvc_ts_stats, on when RVC_TS=1 at creation:
  // every submission (a batch commit or a single-op call) is bracketed by
  // two events, resolved when the stats are read.
  bool ts_on = false;
  long long ts_busy_ns = 0, ts_submits = 0;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> ts_pending;

  Engine();
  ~Engine();

  long long add_buffer(void* p, size_t bytes, size_t block);
  // the block size a buffer of n bytes takes: eight steps per power of two (n
  // itself where it is not pooled)
  static size_t block_size(size_t n);
  void* dev_malloc(size_t bytes);  // hipMalloc, again with the pool emptied where it fails
  void* alloc_block(size_t block);
  void free_block(void* p, size_t block);  // the stream has been waited for
  void drop_oldest();
  void trim_pool();
  void upload(void* dst, const void* src, size_t n);    // may return before the copy has run
  void download(void* dst, const void* src, size_t n);  // waits for the stream
  DevBuf& get(long long id);
  float* fptr(long long id, long long n_floats, const char* what);  // validates size
  void* scratch_for(size_t bytes);
  void sync();
  void ts_collect();  // sync, then fold the pending event pairs into ts_busy_ns
};

// Handle tables (handles are small sequential integers, never raw pointers,
// so a stale or forged handle is rejected instead of dereferenced).
Engine* engine_from_handle(long long h);

}  // namespace rvc
