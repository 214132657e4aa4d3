#include "device.hpp"

#if defined(__SSE2__) && !defined(__HIP_DEVICE_COMPILE__)
#include <emmintrin.h>
#define MC_STREAM_STORES 1
#endif

#include <algorithm>
#include <climits>
#include <cstdlib>
#include <cstring>

#include "mc_common.h"
#include "mchip/kernels.h"

namespace caffe {

// ---------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------

Context& Context::Get() {
  static thread_local Context ctx;
  return ctx;
}

ThreadStream::ThreadStream() {
  HIP_CHECK(hipStreamCreate(&stream));  // default priority
  mchip::watch_process_exit();
}

ThreadStream::~ThreadStream() {
  mchip::ReleaseGuard guard;
  if (guard.allowed()) (void)hipStreamDestroy(stream);
}

Context::Context() : mode_(CPU), device_(0), pool_(std::make_shared<MemoryPool>()) {
  // HIP's per-thread state is made before this object and so outlives it
  if (gpu_available()) (void)hipPeekAtLastError();
}

bool Context::gpu_available() {
  static const bool available = [] {
    int n = 0;
    return hipGetDeviceCount(&n) == hipSuccess && n > 0;
  }();
  return available;
}

void Context::SetMode(DeviceMode mode, int device) {
  if (mode == GPU) {
    CHECK(gpu_available()) << "SetMode(GPU): no HIP device is visible to this process";
    int n = 0;
    HIP_CHECK(hipGetDeviceCount(&n));
    CHECK(device >= 0 && device < n) << "SetMode(GPU): invalid device id " << device << " ("
                                     << n << " device(s) present)";
    if (stream_ && device != device_) {
      Sync();
      stream_.reset();
    }
    HIP_CHECK(hipSetDevice(device));
    device_ = device;
  }
  mode_ = mode;
}

const std::shared_ptr<ThreadStream>& Context::thread_stream() {
  if (!stream_) {
    HIP_CHECK(hipSetDevice(device_));
    stream_ = std::make_shared<ThreadStream>();
  }
  return stream_;
}

void Context::Sync() {
  if (!stream_) return;
  HIP_CHECK(hipStreamSynchronize(stream_->stream));
  stream_->epoch.fetch_add(1);
}

bool GPUAvailable() { return Context::gpu_available(); }

void SetMode(DeviceMode mode, int device) { Context::Get().SetMode(mode, device); }

MemPoolState64 MemPoolGetState64() { return Context::Get().pool()->GetState(); }

MemPoolState MemPoolGetState() {
  const MemPoolState64 s = MemPoolGetState64();
  auto sat = [](long long v) { return v > INT_MAX ? INT_MAX : static_cast<int>(v); };
  MemPoolState r;
  r.gpu_mem = sat(s.gpu_mem);
  r.cpu_mem = sat(s.cpu_mem);
  r.unused_gpu_mem = sat(s.unused_gpu_mem);
  r.unused_cpu_mem = sat(s.unused_cpu_mem);
  return r;
}

void MemPoolClear() {
  Context::Get().Sync();
  Context::Get().pool()->Clear();
  (void)mcReleaseScratch();  // the kernels' own scratch of this thread
}

// ---------------------------------------------------------------------------
// MemoryPool
// ---------------------------------------------------------------------------

namespace {
size_t round_up(size_t v, size_t a) { return (v + a - 1) / a * a; }
}  // namespace

MemoryPool::~MemoryPool() {
  mchip::ReleaseGuard guard;
  if (guard.allowed()) Clear();
}

MemoryPool::Block MemoryPool::RequestHost(size_t size) {
  size = round_up(size ? size : 1, 256);
  {
    std::lock_guard<std::mutex> lk(mu_);
    auto it = free_host_.lower_bound(size);
    if (it != free_host_.end() && it->first <= 2 * size) {
      Block b = it->second;
      free_host_.erase(it);
      host_unused_ -= b.size;
      return b;
    }
  }
  Block b;
  b.size = size;
  b.device = -1;
  if (Context::gpu_available()) {
    // Pinned, so that hipMemcpyAsync is truly asynchronous.
    HIP_CHECK(hipHostMalloc(&b.ptr, size, hipHostMallocDefault));
    b.pinned = true;
  } else {
    b.ptr = std::aligned_alloc(256, size);
    CHECK(b.ptr) << "host allocation of " << size << " bytes failed";
  }
  std::lock_guard<std::mutex> lk(mu_);
  host_total_ += size;
  return b;
}

MemoryPool::Block MemoryPool::RequestDevice(size_t size, int device) {
  size = round_up(size ? size : 1, 256);
  {
    std::lock_guard<std::mutex> lk(mu_);
    auto it = free_dev_.lower_bound(std::make_pair(device, size));
    if (it != free_dev_.end() && it->first.first == device && it->first.second <= 2 * size) {
      Block b = it->second;
      free_dev_.erase(it);
      dev_unused_ -= b.size;
      return b;
    }
  }
  Block b;
  b.size = size;
  b.device = device;
  HIP_CHECK(hipSetDevice(device));
  hipError_t e = hipMalloc(&b.ptr, size);
  if (e != hipSuccess) {
    // Give cached blocks back and retry once before failing.
    (void)hipGetLastError();
    Clear();
    e = hipMalloc(&b.ptr, size);
  }
  CHECK(e == hipSuccess) << "hipMalloc(" << size << " bytes): " << hipGetErrorString(e);
  mchip::watch_process_exit();
  std::lock_guard<std::mutex> lk(mu_);
  dev_total_ += size;
  return b;
}

void MemoryPool::Return(const Block& b) {
  if (!b.ptr) return;
  std::lock_guard<std::mutex> lk(mu_);
  if (b.device < 0) {
    free_host_.insert(std::make_pair(b.size, b));
    host_unused_ += b.size;
  } else {
    free_dev_.insert(std::make_pair(std::make_pair(b.device, b.size), b));
    dev_unused_ += b.size;
  }
}

void MemoryPool::Clear() {
  std::lock_guard<std::mutex> lk(mu_);
  for (auto& kv : free_host_) {
    if (kv.second.pinned) (void)hipHostFree(kv.second.ptr);
    else std::free(kv.second.ptr);
    host_total_ -= kv.second.size;
  }
  for (auto& kv : free_dev_) {
    (void)hipFree(kv.second.ptr);
    dev_total_ -= kv.second.size;
  }
  free_host_.clear();
  free_dev_.clear();
  host_unused_ = 0;
  dev_unused_ = 0;
}

MemPoolState64 MemoryPool::GetState() {
  std::lock_guard<std::mutex> lk(mu_);
  MemPoolState64 s;
  s.gpu_mem = dev_total_;
  s.cpu_mem = host_total_;
  s.unused_gpu_mem = dev_unused_;
  s.unused_cpu_mem = host_unused_;
  return s;
}

// ---------------------------------------------------------------------------
// SyncedMemory
// ---------------------------------------------------------------------------

SyncedMemory::SyncedMemory(size_t size)
    : size_(size), head_(UNINITIALIZED), pool_(Context::Get().pool()), version_(0),
      h2d_epoch_(0) {}

SyncedMemory::~SyncedMemory() {
  // A pinned block that still feeds an asynchronous upload must not be recycled.
  try {
    wait_pending_h2d();
  } catch (...) {
  }
  pool_->Return(host_);
  pool_->Return(dev_);
}

void SyncedMemory::set_pending_h2d() {
  h2d_stream_ = Context::Get().thread_stream();
  h2d_epoch_ = h2d_stream_->epoch.load();
}

void SyncedMemory::wait_pending_h2d() {
  if (!h2d_stream_) return;
  if (h2d_stream_->epoch.load() == h2d_epoch_) HIP_CHECK(hipStreamSynchronize(h2d_stream_->stream));
  h2d_stream_.reset();
}

void SyncedMemory::to_cpu() {
  switch (head_) {
    case UNINITIALIZED:
      host_ = pool_->RequestHost(size_);
      head_ = HEAD_AT_CPU;
      break;
    case HEAD_AT_GPU: {
      if (!host_.ptr) host_ = pool_->RequestHost(size_);
      Context& ctx = Context::Get();
      HIP_CHECK(hipMemcpyAsync(host_.ptr, dev_.ptr, size_, hipMemcpyDeviceToHost, ctx.stream()));
      ctx.Sync();
      head_ = SYNCED;
      break;
    }
    case HEAD_AT_CPU:
    case SYNCED:
      break;
  }
}

void SyncedMemory::to_gpu() {
  CHECK(Context::gpu_available()) << "device memory requested but no HIP device is present";
  switch (head_) {
    case UNINITIALIZED:
      dev_ = pool_->RequestDevice(size_, Context::Get().device());
      head_ = HEAD_AT_GPU;
      break;
    case HEAD_AT_CPU: {
      if (!dev_.ptr) dev_ = pool_->RequestDevice(size_, Context::Get().device());
      Context& ctx = Context::Get();
      HIP_CHECK(hipMemcpyAsync(dev_.ptr, host_.ptr, size_, hipMemcpyHostToDevice, ctx.stream()));
      set_pending_h2d();
      head_ = SYNCED;
      break;
    }
    case HEAD_AT_GPU:
    case SYNCED:
      // an upload queued by another thread (Assign) is not ordered before this thread's launches
      if (h2d_stream_ && h2d_stream_ != Context::Get().thread_stream()) wait_pending_h2d();
      break;
  }
}

const void* SyncedMemory::cpu_data() {
  to_cpu();
  return host_.ptr;
}

void* SyncedMemory::mutable_cpu_data() {
  to_cpu();
  wait_pending_h2d();  // the caller is about to overwrite the upload's source
  head_ = HEAD_AT_CPU;
  ++version_;
  return host_.ptr;
}

const void* SyncedMemory::gpu_data() {
  to_gpu();
  return dev_.ptr;
}

void* SyncedMemory::mutable_gpu_data() {
  to_gpu();
  head_ = HEAD_AT_GPU;
  ++version_;
  return dev_.ptr;
}

namespace {
// memcpy to memory that the processor will not read again, `to` aligned to 64 bytes: stores
// that go past its caches spare reading every line of the destination first and leave the
// link's reads to memory (one core, 38 MB: 31-35 GB/s with memmove, 39-46 so).
void stream_copy(char* to, const char* from, size_t bytes) {
  size_t i = 0;
#ifdef MC_STREAM_STORES
  for (; i + 64 <= bytes; i += 64) {
    const __m128i a = _mm_loadu_si128(reinterpret_cast<const __m128i*>(from + i));
    const __m128i b = _mm_loadu_si128(reinterpret_cast<const __m128i*>(from + i + 16));
    const __m128i c = _mm_loadu_si128(reinterpret_cast<const __m128i*>(from + i + 32));
    const __m128i d = _mm_loadu_si128(reinterpret_cast<const __m128i*>(from + i + 48));
    _mm_stream_si128(reinterpret_cast<__m128i*>(to + i), a);
    _mm_stream_si128(reinterpret_cast<__m128i*>(to + i + 16), b);
    _mm_stream_si128(reinterpret_cast<__m128i*>(to + i + 32), c);
    _mm_stream_si128(reinterpret_cast<__m128i*>(to + i + 48), d);
  }
  _mm_sfence();  // before the copy engine is told to read it
#endif
  std::memcpy(to + i, from + i, bytes - i);
}
}  // namespace

// A large blob goes to pinned memory a piece at a time, each piece on its way to the device
// while the next one is copied; a host copy of the whole blob first leaves the copy engine
// waiting (batch of 64 images, 38.5 MB: 6.25 ms per ResNet-50 pass, 5.47 in pieces of 2 MiB,
// 5.1 with streaming stores and a first piece of 512 KiB, which the engine waits for).
// Only for all of the block: a part would leave the two copies different behind it.  (A blob
// that has been larger keeps its larger block, so later, smaller arrays are copied whole and
// uploaded by the forward.)
void SyncedMemory::Assign(const void* src, size_t bytes) {
  CHECK_LE(bytes, size_) << "SyncedMemory::Assign: more bytes than the block holds";
  Context& ctx = Context::Get();
  if (bytes != size_ || ctx.mode() != GPU || !Context::gpu_available()) {
    std::memmove(mutable_cpu_data(), src, bytes);
    return;
  }
  wait_pending_h2d();
  if (!host_.ptr) host_ = pool_->RequestHost(size_);
  if (!dev_.ptr) dev_ = pool_->RequestDevice(size_, ctx.device());
  head_ = HEAD_AT_CPU;  // what holds if a copy below fails
  ++version_;
  const char* from = static_cast<const char*>(src);
  char* const to = static_cast<char*>(host_.ptr);
  const bool apart = from + bytes <= to || to + bytes <= from;
  // (up to 2 MiB in one piece and with ordinary stores: a second copy costs more than it hides,
  // 64 x 56 x 56 137 us per pass in two, 132 in one)
  const size_t largest = size_t(2) << 20;
  const bool stream = apart && bytes > largest;
  size_t piece = bytes > 2 * largest ? largest / 4 : largest;
  for (size_t off = 0; off < bytes; off += piece, piece = std::min(2 * piece, largest)) {
    if (off > 0 && bytes - off < piece + piece / 2) piece = bytes - off;  // no short last piece
    const size_t n = std::min(piece, bytes - off);
    char* host = to + off;
    if (stream) {
      stream_copy(host, from + off, n);
    } else {
      std::memmove(host, from + off, n);
    }
    HIP_CHECK(hipMemcpyAsync(static_cast<char*>(dev_.ptr) + off, host, n, hipMemcpyHostToDevice, ctx.stream()));
    set_pending_h2d();
  }
  head_ = SYNCED;
}

}  // namespace caffe

extern "C" void* mcCurrentStream(void) {
  try {
    return caffe::Context::Get().stream();
  } catch (const caffe::Error&) {
    return nullptr;
  }
}
