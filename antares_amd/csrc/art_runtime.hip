// Device runtime of libantares_amd.so: initialisation, in-process compilation
// of generated HIP source, code-object loading, kernel launch and timing.
// This is the counterpart of the reference's `namespace ab` for HIP
// (backends/c-rocm/include/backend.hpp:46-253) behind a flat C ABI.
#include <hip/hiprtc.h>
#include <string.h>

#include <mutex>
#include <vector>

#include "art_common.h"

namespace art {

std::string& last_error() {
  static thread_local std::string e;
  return e;
}

int fail(const char* fmt, ...) {
  char buf[2048];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  last_error() = buf;
  return 1;
}

static constexpr int kMaxDevices = 16;
// 64 MiB: split-K accumulators, partial tiles of the split-K GEMM and tile states of the scan kernels.
static constexpr size_t kWorkspaceBytes = 64u << 20;
struct StreamWorkspace {
  hipStream_t stream;
  Workspace ws;
};
struct DeviceState {
  bool initialised = false;
  int used = 0;
  StreamWorkspace slot[kMaxStreamsPerDevice];
};
static DeviceState g_dev[kMaxDevices];
static std::mutex g_mu;

int compute_units() {
  static int cached[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}

static int allocate_workspace(Workspace* ws) {
  ART_HIP(hipMalloc(&ws->base, kWorkspaceBytes));
  hipError_t e = hipMemset(ws->base, 0, kWorkspaceBytes);
  if (e == hipSuccess) e = hipDeviceSynchronize();        // the zeroes are in place before any stream uses them
  if (e != hipSuccess) {
    (void)hipFree(ws->base);
    ws->base = nullptr;
    return fail("zeroing the workspace failed: %s", hipGetErrorString(e));
  }
  ws->bytes = kWorkspaceBytes;
  return 0;
}

Workspace* workspace(hipStream_t stream) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fail("workspace: no current device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_mu);
  DeviceState& d = g_dev[dev];
  if (!d.initialised) {
    fail("call art_init first");
    return nullptr;
  }
  int free_slot = -1;
  for (int i = 0; i < d.used; ++i) {
    if (d.slot[i].ws.base != nullptr && d.slot[i].stream == stream) return &d.slot[i].ws;
    if (d.slot[i].ws.base == nullptr && free_slot < 0) free_slot = i;        // released by art_release_stream
  }
  if (free_slot < 0 && d.used == kMaxStreamsPerDevice) {
    fail("more than %d streams use split-K / two-pass kernels on device %d; order them on fewer streams, or hand the "
         "workspaces of destroyed streams back with art_release_stream", kMaxStreamsPerDevice, dev);
    return nullptr;
  }
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    fail("the first split-K / two-pass launch on a stream allocates its workspace and cannot be captured into a graph: "
         "run the operator once on this stream before capturing");
    return nullptr;
  }
  StreamWorkspace& sw = d.slot[free_slot >= 0 ? free_slot : d.used];
  sw.stream = stream;
  sw.ws = Workspace{};
  if (allocate_workspace(&sw.ws)) return nullptr;
  if (free_slot < 0) ++d.used;
  return &sw.ws;
}

// Frees the workspace of (current device, stream) after the stream's work has finished; the slot can be taken by
// another stream afterwards.  A stream without a workspace is no error.
int release_stream(hipStream_t stream) {
  int dev = 0;
  ART_HIP(hipGetDevice(&dev));
  ART_REQUIRE(dev >= 0 && dev < kMaxDevices, "art_release_stream: bad device %d", dev);
  ART_REQUIRE(stream != nullptr, "art_release_stream: the default stream keeps its workspace");
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    DeviceState& d = g_dev[dev];
    for (int i = 0; i < d.used; ++i)
      if (d.slot[i].ws.base != nullptr && d.slot[i].stream == stream) {
        base = d.slot[i].ws.base;
        d.slot[i].ws = Workspace{};
        d.slot[i].stream = nullptr;
      }
  }
  if (base == nullptr) return 0;
  ART_HIP(hipStreamSynchronize(stream));       // outside the lock: launches on other streams go on meanwhile
  ART_HIP(hipFree(base));
  return 0;
}

static std::string& compile_log() {
  static thread_local std::string s;
  return s;
}

}  // namespace art

struct art_module {
  hipModule_t handle;
};
struct art_func {
  hipFunction_t handle;
};

extern "C" {

const char* art_last_error(void) { return art::last_error().c_str(); }
const char* art_compile_log(void) { return art::compile_log().c_str(); }
size_t art_workspace_bytes(void) { return art::kWorkspaceBytes; }
int art_release_stream(void* stream) { return art::release_stream((hipStream_t)stream); }

int art_init(int device) {
  int count = 0;
  ART_HIP(hipGetDeviceCount(&count));
  ART_REQUIRE(device >= 0 && device < count && device < art::kMaxDevices, "art_init: no such device %d (have %d)", device, count);
  ART_HIP(hipSetDevice(device));
  {
    std::lock_guard<std::mutex> lock(art::g_mu);
    art::g_dev[device].initialised = true;
  }
  if (art::gemv_noalloc_setup(device)) return 1;
  // the workspace of the default stream now; other streams get theirs when they first need one
  return art::workspace(nullptr) ? 0 : 1;
}

int art_device_props(art_props* out) {
  ART_REQUIRE(out != nullptr, "art_device_props: null output");
  int dev = 0;
  ART_HIP(hipGetDevice(&dev));
  hipDeviceProp_t p;
  ART_HIP(hipGetDeviceProperties(&p, dev));
  memset(out, 0, sizeof(*out));
  snprintf(out->name, sizeof(out->name), "%s", p.name);
  snprintf(out->arch, sizeof(out->arch), "%s", p.gcnArchName);
  if (char* colon = strchr(out->arch, ':')) *colon = 0;
  out->compute_units = p.multiProcessorCount;
  out->wavefront_size = p.warpSize;
  out->max_threads_per_block = p.maxThreadsPerBlock;
  out->lds_bytes_per_block = (int)p.sharedMemPerBlock;
  out->clock_khz = p.clockRate;
  out->memory_clock_khz = p.memoryClockRate;
  out->memory_bus_width_bits = p.memoryBusWidth;
  out->l2_bytes = p.l2CacheSize;
  out->total_memory_bytes = p.totalGlobalMem;
  return 0;
}

// Of every kernel that art_module_compile makes: packed-FP32 instruction selection is switched off, the first arguments start in registers.
#define ART_COMPILE_OPTIONS(X)                                                                                                       \
  X("-O3") X("-std=c++17") X("-Wno-ignored-attributes") X("-Xclang") X("-target-feature") X("-Xclang") X("-packed-fp32-ops") X("-mllvm") \
  X("-amdgpu-kernarg-preload-count=14")
#define ART_OPTION_TEXT(option) option " "
#define ART_OPTION_ITEM(option) , option
const char* art_compile_options(void) { return ART_COMPILE_OPTIONS(ART_OPTION_TEXT); }

int art_module_compile(const char* hip_source, const char* arch, void** blob, size_t* size) {
  ART_REQUIRE(hip_source && blob && size, "art_module_compile: null argument");
  art::compile_log().clear();
  hiprtcProgram prog;
  hiprtcResult r = hiprtcCreateProgram(&prog, hip_source, "autort_kernel.hip", 0, nullptr, nullptr);
  ART_REQUIRE(r == HIPRTC_SUCCESS, "hiprtcCreateProgram: %s", hiprtcGetErrorString(r));
  std::string arch_opt = std::string("--offload-arch=") + ((arch && *arch) ? arch : "gfx950");
  const char* opts[] = {arch_opt.c_str() ART_COMPILE_OPTIONS(ART_OPTION_ITEM)};
  r = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
  size_t log_size = 0;
  hiprtcGetProgramLogSize(prog, &log_size);
  if (log_size > 1) {
    art::compile_log().resize(log_size);
    hiprtcGetProgramLog(prog, &art::compile_log()[0]);
  }
  if (r != HIPRTC_SUCCESS) {
    hiprtcDestroyProgram(&prog);
    return art::fail("compilation failed: %s\n%s", hiprtcGetErrorString(r), art::compile_log().c_str());
  }
  size_t n = 0;
  hiprtcGetCodeSize(prog, &n);
  void* mem = malloc(n);
  if (!mem) {
    hiprtcDestroyProgram(&prog);
    return art::fail("art_module_compile: out of host memory");
  }
  hiprtcGetCode(prog, (char*)mem);
  hiprtcDestroyProgram(&prog);
  *blob = mem;
  *size = n;
  return 0;
}

void art_blob_free(void* blob) { free(blob); }

int art_module_load(const void* image, size_t size, art_module** out) {
  ART_REQUIRE(image && size > 0 && out, "art_module_load: null argument");
  hipModule_t m;
  ART_HIP(hipModuleLoadData(&m, image));
  *out = new art_module{m};
  return 0;
}

int art_module_load_file(const char* path, art_module** out) {
  ART_REQUIRE(path && out, "art_module_load_file: null argument");
  FILE* f = fopen(path, "rb");
  if (!f) return art::fail("art_module_load_file: cannot open %s", path);
  std::vector<char> image;
  char buf[65536];
  size_t n;
  while ((n = fread(buf, 1, sizeof(buf), f)) > 0) image.insert(image.end(), buf, buf + n);
  fclose(f);
  ART_REQUIRE(!image.empty(), "art_module_load_file: %s is empty", path);
  return art_module_load(image.data(), image.size(), out);
}

int art_module_unload(art_module* module) {
  ART_REQUIRE(module != nullptr, "art_module_unload: null module");
  ART_HIP(hipModuleUnload(module->handle));
  delete module;
  return 0;
}

int art_get_function(art_module* module, const char* name, art_func** out) {
  ART_REQUIRE(module && name && out, "art_get_function: null argument");
  hipFunction_t f;
  hipError_t e = hipModuleGetFunction(&f, module->handle, name);
  if (e != hipSuccess) return art::fail("kernel `%s` not found in module: %s", name, hipGetErrorString(e));
  *out = new art_func{f};
  return 0;
}

int art_launch(art_func* func, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz,
               unsigned lds_bytes, void* stream, const uint64_t* args, int nargs) {
  ART_REQUIRE(func != nullptr, "art_launch: null function");
  ART_REQUIRE(nargs >= 0 && nargs <= 64, "art_launch: bad argument count %d", nargs);
  ART_REQUIRE(bx * by * bz >= 1 && bx * by * bz <= 1024, "art_launch: bad block %ux%ux%u", bx, by, bz);
  if (gx == 0 || gy == 0 || gz == 0) return 0;   // empty iteration space: nothing to run
  void* params[64];
  for (int i = 0; i < nargs; ++i) params[i] = (void*)&args[i];
  ART_HIP(hipModuleLaunchKernel(func->handle, gx, gy, gz, bx, by, bz, lds_bytes, (hipStream_t)stream, params, nullptr));
  return 0;
}

int art_event_create(void** event) {
  ART_REQUIRE(event != nullptr, "art_event_create: null output");
  hipEvent_t e;
  ART_HIP(hipEventCreate(&e));
  *event = e;
  return 0;
}
int art_event_record(void* event, void* stream) {
  ART_HIP(hipEventRecord((hipEvent_t)event, (hipStream_t)stream));
  return 0;
}
int art_event_elapsed_ms(void* start, void* stop, float* ms) {
  ART_REQUIRE(ms != nullptr, "art_event_elapsed_ms: null output");
  ART_HIP(hipEventSynchronize((hipEvent_t)stop));
  ART_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop));
  return 0;
}
int art_event_destroy(void* event) {
  ART_HIP(hipEventDestroy((hipEvent_t)event));
  return 0;
}
int art_stream_synchronize(void* stream) {
  ART_HIP(hipStreamSynchronize((hipStream_t)stream));
  return 0;
}

}  // extern "C"

// ------------------------------------------------------------ copy kernel
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void art_copy_kernel(u32x4* __restrict__ dst, const u32x4* __restrict__ src, size_t nvec) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * 256;
  for (; i < nvec; i += stride) dst[i] = __builtin_nontemporal_load(&src[i]);
}

extern "C" int art_copy_bytes(void* dst_dev, const void* src_dev, size_t bytes, void* stream) {
  ART_REQUIRE(((uintptr_t)dst_dev % 16) == 0 && ((uintptr_t)src_dev % 16) == 0 && bytes % 16 == 0,
              "art_copy_bytes: pointers and size must be multiples of 16");
  size_t nvec = bytes / 16;
  if (nvec == 0) return 0;
  size_t blocks = (nvec + 255) / 256;
  if (blocks > 256 * 16) blocks = 256 * 16;
  art_copy_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>((u32x4*)dst_dev, (const u32x4*)src_dev, nvec);
  ART_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------ read-only kernel
// The access pattern of the weight stream of the int4 GEMV with nothing behind it: a block of 256 threads owns 32 KiB,
// every thread issues its eight 16-byte loads (128 contiguous bytes per 8 lanes, rows `pitch` bytes apart) before it
// looks at any of them, and the block leaves one word that depends on all of them.  What this takes for a buffer is
// what a single dependent launch spends on getting the bytes on chip, whatever arithmetic follows.
__global__ __launch_bounds__(256) void art_read_kernel(const unsigned char* __restrict__ src, size_t pitch, int tiles,
                                                       unsigned int* __restrict__ sink) {
  const int tid = threadIdx.x, cl = tid & 7, kl = tid >> 3;
  const int tile = blockIdx.x % tiles, split = blockIdx.x / tiles;
  const unsigned char* p = src + ((size_t)split * 256 + (size_t)kl * 8) * pitch + (size_t)tile * 128 + cl * 16;
  u32x4 w[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) w[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + (size_t)i * pitch));
  unsigned int acc = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) acc ^= w[i][0] ^ w[i][1] ^ w[i][2] ^ w[i][3];
  if (acc == 0x9E3779B9u) sink[blockIdx.x] = acc;        // (almost) never true: the loads stay, the stores do not happen
}

extern "C" int art_read_bytes(const void* src_dev, size_t bytes, void* sink_dev, void* stream) {
  // viewed as rows of 11008 bytes when the size allows it (the headline weight matrix), else rows of 128 bytes
  ART_REQUIRE(src_dev && sink_dev && ((uintptr_t)src_dev % 16) == 0 && bytes % 32768 == 0 && bytes > 0,
              "art_read_bytes: need a 16-byte aligned buffer of a multiple of 32768 bytes");
  const size_t pitch = (bytes % (11008u * 256u) == 0) ? 11008 : 128;
  const int tiles = (int)(pitch / 128);
  const size_t blocks = bytes / 32768;
  ART_REQUIRE(blocks <= 4096, "art_read_bytes: at most 128 MiB per launch (sink has 4096 words)");
  art_read_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>((const unsigned char*)src_dev, pitch, tiles,
                                                                               (unsigned int*)sink_dev);
  ART_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------ store-only kernel
// The counterpart of the read-only launch for writes: every thread stores 16-byte vectors of a constant with
// non-temporal stores, nothing is read.  What it takes is the floor of a launch that has to write these bytes.
__global__ __launch_bounds__(256) void art_fill_kernel(u32x4* __restrict__ dst, size_t nvec, unsigned int value) {
  size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * 256;
  const u32x4 v = {value, value, value, value};
  for (; i < nvec; i += stride) __builtin_nontemporal_store(v, &dst[i]);
}

extern "C" int art_fill_bytes(void* dst_dev, size_t bytes, unsigned int value, void* stream) {
  ART_REQUIRE(dst_dev && ((uintptr_t)dst_dev % 16) == 0 && bytes % 16 == 0, "art_fill_bytes: pointer and size must be multiples of 16");
  const size_t nvec = bytes / 16;
  if (nvec == 0) return 0;
  size_t blocks = (nvec + 255) / 256;
  if (blocks > 256 * 16) blocks = 256 * 16;
  art_fill_kernel<<<dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream>>>((u32x4*)dst_dev, nvec, value);
  ART_LAUNCH_CHECK();
  return 0;
}

// ------------------------------------------------------------ phases inside one launch
// What a grid-wide barrier inside a kernel costs on this part, and whether a persistent kernel can keep the weight
// stream going across it: 256 resident blocks run `phases` phases; in a phase every block fetches its share of
// `phase_bytes` with the read-only launch's pattern (three 32 KiB units per block at most) and then all blocks meet.
// The meeting uses no atomics and no fences: a block's thirteenth wavefront stores (phase, launch tag) into the
// block's own word with an agent-scope store and polls everybody's words with agent-scope loads, a bounded number
// of times; the twelve worker wavefronts wait at an LDS-only barrier, so loads they have in flight stay in flight.
//   mode 0: no loads at all (the barrier by itself);  mode 1: a phase's loads are issued after the previous barrier;
//   mode 2: the NEXT phase's loads are issued before the barrier (what a persistent decode kernel would do).
constexpr int kChainBlocks = 256, kChainWorkers = 768, kChainThreads = 832, kChainSpinLimit = 1 << 18;

__global__ __launch_bounds__(kChainThreads) void art_phase_chain_kernel(const unsigned char* __restrict__ src, size_t phase_bytes,
                                                                        int phases, size_t pitch, int tiles, int mode,
                                                                        unsigned long long* __restrict__ exchange,
                                                                        unsigned int* __restrict__ sink,
                                                                        unsigned int* __restrict__ status) {
  __shared__ int s_ok;
  __shared__ unsigned long long s_tag;
  const int tid = threadIdx.x, lane = tid & 63, q = tid >> 8, t = tid & 255, cl = t & 7, kl = t >> 3;
  const bool control = tid >= kChainWorkers;
  unsigned long long* launches = exchange;
  unsigned long long* words = exchange + 8;
  if (tid == kChainWorkers) s_tag = __hip_atomic_load(launches, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  const int units = (int)(phase_bytes / 32768);
  const int unit = (int)blockIdx.x + kChainBlocks * q;
  const bool has = !control && unit < units;
  const int tile = unit % tiles, split = unit / tiles;
  const size_t off = has ? ((size_t)split * 256 + (size_t)kl * 8) * pitch + (size_t)tile * 128 + cl * 16 : 0;
  __syncthreads();
  const unsigned long long tag = s_tag;
  unsigned int acc = 0;
  u32x4 w[8];
  if (mode == 2 && has) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(src + off + (size_t)i * pitch));
  }
  for (int ph = 0; ph < phases; ++ph) {
    if (mode == 1 && has) {
      const unsigned char* p = src + (size_t)ph * phase_bytes + off;
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + (size_t)i * pitch));
    }
    if (mode != 0 && has) {
#pragma unroll
      for (int i = 0; i < 8; ++i) acc ^= w[i][0] ^ w[i][1] ^ w[i][2] ^ w[i][3];
    }
    if (mode == 2 && has && ph + 1 < phases) {
      const unsigned char* p = src + (size_t)(ph + 1) * phase_bytes + off;
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p + (size_t)i * pitch));
    }
    // ---- all blocks meet
    art_lds_barrier();                       // every wavefront of the block has finished the phase
    if (control) {
      const unsigned long long want = (tag << 16) | (unsigned long long)(ph + 1);
      if (lane == 0) __hip_atomic_store(words + blockIdx.x, want, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      bool done = false;
      for (int spin = 0; spin < kChainSpinLimit && !done; ++spin) {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < kChainBlocks / 64; ++k)
          ok = ok && __hip_atomic_load(words + lane + 64 * k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= want;
        done = __all(ok);
      }
      if (lane == 0) {
        s_ok = done ? 1 : 0;
        if (!done) __hip_atomic_store(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    art_lds_barrier();
    if (!s_ok) break;                        // a block that gave up stops meeting; the others give up in turn and exit
  }
  if (blockIdx.x == 0 && tid == kChainWorkers)   // the next launch on this workspace gets a new tag
    __hip_atomic_store(launches, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (acc == 0x9E3779B9u) sink[blockIdx.x] = acc;
}

extern "C" int art_phase_chain_probe(const void* src_dev, size_t src_bytes, size_t phase_bytes, int phases, int mode, void* sink_dev,
                                     void* status_dev, void* stream) {
  ART_REQUIRE(src_dev && sink_dev && status_dev && ((uintptr_t)src_dev % 16) == 0, "art_phase_chain_probe: null or misaligned pointer");
  ART_REQUIRE(mode >= 0 && mode <= 2 && phases >= 1 && phases <= 65535, "art_phase_chain_probe: mode 0..2, 1..65535 phases");
  ART_REQUIRE(phase_bytes > 0 && phase_bytes % 32768 == 0 && phase_bytes / 32768 <= 3 * (size_t)kChainBlocks,
              "art_phase_chain_probe: a phase is a multiple of 32768 bytes, at most %d", 3 * kChainBlocks * 32768);
  ART_REQUIRE((size_t)phases * phase_bytes <= src_bytes, "art_phase_chain_probe: %d phases of %zu bytes do not fit the %zu bytes of src", phases,
              phase_bytes, src_bytes);
  ART_REQUIRE(art::compute_units() >= kChainBlocks, "art_phase_chain_probe: needs %d compute units (all blocks must be resident)", kChainBlocks);
  art::Workspace* wsp = art::workspace((hipStream_t)stream);
  if (!wsp) return 1;
  const size_t pitch = (phase_bytes % (11008u * 256u) == 0) ? 11008 : 128;
  art_phase_chain_kernel<<<dim3(kChainBlocks), dim3(kChainThreads), 0, (hipStream_t)stream>>>(
      (const unsigned char*)src_dev, phase_bytes, phases, pitch, (int)(pitch / 128), mode,
      reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(wsp->base) + art::kExchangeOffset), (unsigned int*)sink_dev,
      (unsigned int*)status_dev);
  ART_LAUNCH_CHECK();
  return 0;
}

// ---- device memory for callers that own no allocator (the reference's evaluator; the torch plugin uses torch's)
extern "C" int art_alloc(size_t bytes, void** out_dev) {
  ART_REQUIRE(out_dev != nullptr, "art_alloc: null output");
  *out_dev = nullptr;
  if (bytes == 0) return 0;
  ART_HIP(hipMalloc(out_dev, bytes));
  return 0;
}

extern "C" int art_free(void* dev) {
  if (dev) ART_HIP(hipFree(dev));
  return 0;
}

extern "C" int art_memcpy_htod(void* dst_dev, const void* src_host, size_t bytes, void* stream) {
  if (bytes) ART_HIP(hipMemcpyAsync(dst_dev, src_host, bytes, hipMemcpyHostToDevice, (hipStream_t)stream));
  return 0;
}

extern "C" int art_memcpy_dtod(void* dst_dev, const void* src_dev, size_t bytes, void* stream) {
  if (bytes) ART_HIP(hipMemcpyAsync(dst_dev, src_dev, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream));
  return 0;
}

extern "C" int art_memcpy_dtoh(void* dst_host, const void* src_dev, size_t bytes, void* stream) {
  if (bytes) ART_HIP(hipMemcpyAsync(dst_host, src_dev, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream));
  return 0;
}
