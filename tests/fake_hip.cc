// fake_hip.cc -- a HIP runtime without a GPU, for tests of the host side of the
// C ABI: device memory is host memory, streams and events are nothing, and
// kernels are not run but noted (name, grid, block).  Loaded into the global
// scope before the library, whose HIP calls then come here (tests/fake_hip.py).
#include <cxxabi.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "lgpu_kernels.h"

namespace {

struct Config {
   dim3 grid, block;
   size_t shared;
   hipStream_t stream;
};

std::vector<Config> configs;
std::map<const void *, std::string> kernels; // host stub -> demangled name
std::map<char *, size_t> live, pinned;       // device allocations, hipHostMalloc
std::string launches, report;
long mallocsLeft = -1; // hipMalloc fails once this many have succeeded (< 0: never)
long copies = 0, capturing = 0;
std::vector<lgpu::EosSlot> eosSlots; // of the last k_eos launch

bool holds(const std::map<char *, size_t> &blocks, const void *p)
{
   auto it = blocks.upper_bound((char *)p);
   return it != blocks.begin() && (--it, (const char *)p < it->first + it->second);
}
bool device_pointer(const void *p) { return holds(live, p); }

} // namespace

extern "C" {

// --- what the tests read ---
// "name grid block" of every launch since the last call, one a line
const char *fake_launches()
{
   report.swap(launches);
   launches.clear();
   return report.c_str();
}
void fake_fail_malloc_after(long n) { mallocsLeft = n; }
long fake_copies() { return copies; } // hipMemcpy calls
int fake_eos_slots(const lgpu::EosSlot **slots)
{
   *slots = eosSlots.data();
   return (int)eosSlots.size();
}

// --- registration and launch ---
void **__hipRegisterFatBinary(const void *)
{
   static void *handle;
   return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
   int status = 0;
   char *plain = abi::__cxa_demangle(name, nullptr, nullptr, &status);
   kernels[host] = status == 0 ? plain : name;
   std::free(plain);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
   configs.push_back({grid, block, shared, stream});
   return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream)
{
   *grid = configs.back().grid;
   *block = configs.back().block;
   *shared = configs.back().shared;
   *stream = configs.back().stream;
   configs.pop_back();
   return hipSuccess;
}
hipError_t hipLaunchKernel(const void *host, dim3 grid, dim3 block, void **args, size_t, hipStream_t)
{
   std::string name = kernels[host];
   const char *const anonymous = "(anonymous namespace)::";
   if (const size_t at = name.find(anonymous); at != std::string::npos) name.erase(at, std::strlen(anonymous));
   name = name.substr(0, name.find('('));
   // an ensemble's brick kernels: their tables have to be allocated, and made
   // for the kernel and the grid
   if (name.find("k_nodal_b") != std::string::npos || name.find("k_kin_b") != std::string::npos ||
       name.find("k_kin_f") != std::string::npos) {
      const lgpu::DevState &s = *static_cast<const lgpu::DevState *>(args[0]);
      if (s.nMembers) {
         const bool nodal = name.find("k_nodal") != std::string::npos;
         const lgpu::MemberBlock *blocks = nodal ? s.nodalBlocks : s.kinBlocks;
         const bool walk = name.find("_brick") != std::string::npos;
         if (!device_pointer(s.memberBrick) || !device_pointer(blocks) || !device_pointer(blocks + grid.x - 1))
            name += "!freed-tables";
         else
            for (unsigned i = 0; i < grid.x; ++i) {
               const lgpu::Brick &g = s.memberBrick[blocks[i].member].g;
               const int64_t n = nodal ? (walk ? (int64_t)g.tilesX * g.tilesY * g.chunks
                                               : (int64_t)g.blkX * g.blkY * g.blkZ)
                                       : (walk ? (int64_t)g.kinTilesX * g.kinTilesY * g.kinChunks
                                               : ((int64_t)g.s * g.s * g.s + 255) / 256);
               const bool lastOfMember = i + 1 == grid.x || blocks[i + 1].member != blocks[i].member;
               if ((int64_t)blocks[i].wg >= n || (!walk && lastOfMember && (int64_t)blocks[i].wg + 1 != n)) {
                  name += "!other-tables";
                  break;
               }
            }
      }
   }
   if (name.find("k_eos<") != std::string::npos) {
      const lgpu::DevState &s = *static_cast<const lgpu::DevState *>(args[0]);
      eosSlots.assign(s.eosSlot, s.eosSlot + grid.x);
   }
   launches += name + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + "\n";
   return hipSuccess;
}

// --- device: 256 CUs, the occupancies of the step kernels ---
hipError_t hipGetDevice(int *dev)
{
   *dev = 0;
   return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *value, hipDeviceAttribute_t what, int)
{
   *value = what == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
   return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *host)
{
   *a = hipFuncAttributes{};
   const std::string &name = kernels[host];
   const bool mixed = name.find("PolicyMixed") != std::string::npos;
   const bool nodal = name.find("k_nodal_brick") != std::string::npos;
   a->numRegs = nodal && !mixed ? 256 : 168;
   a->sharedSizeBytes = nodal ? (mixed ? 36864 : 73728) : 49000;
   return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }

// --- memory ---
hipError_t hipMalloc(void **p, size_t bytes)
{
   if (mallocsLeft == 0) return hipErrorOutOfMemory;
   if (mallocsLeft > 0) --mallocsLeft;
   *p = std::calloc(1, bytes ? bytes : 1);
   live[(char *)*p] = bytes;
   return hipSuccess;
}
hipError_t hipFree(void *p)
{
   live.erase((char *)p);
   std::free(p);
   return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
   *p = std::calloc(1, bytes);
   pinned[(char *)*p] = bytes;
   return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
   *a = hipPointerAttribute_t{};
   a->type = holds(pinned, p) ? hipMemoryTypeHost : hipMemoryTypeDevice;
   return holds(pinned, p) || device_pointer(p) ? hipSuccess : hipErrorInvalidValue;
}
hipError_t hipHostFree(void *p)
{
   pinned.erase((char *)p);
   std::free(p);
   return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind)
{
   ++copies;
   std::memcpy(dst, src, bytes);
   return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t)
{
   std::memcpy(dst, src, bytes);
   return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t bytes)
{
   std::memset(p, v, bytes);
   return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
   *p = nullptr;
   return hipErrorUnknown;
}

// --- streams, events (1 ms apart), graphs (launched once, when captured) ---
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
   *s = (hipStream_t)&copies;
   return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e)
{
   *e = (hipEvent_t)&copies;
   return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
   *ms = 1.f;
   return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
   *g = (hipGraph_t)&capturing;
   return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
   *x = (hipGraphExec_t)&capturing;
   return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

} // extern "C"
