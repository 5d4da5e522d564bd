// pf_noalloc.hip — pf_gpu_diffusion_solver_noalloc: the diffusion-only offload of
// pf_gpu_diffusion_solver (GPU_Diffusion_solver, gpu_solver.cpp:204-218) for callers that cannot
// allocate device memory (code under HIP graph capture, serving loops, harnesses that forbid
// hipMalloc).  The caller passes value_phase and total_conc in device memory and a stream; the
// sub-steps run asynchronously on that stream with the kernels of the handle API: the bulk flags and
// the list once per call, then the tile kernel (one plane, several sub-steps per launch) or the
// one-launch sub-step (3D; large domains the LDS-tiled full formula where no phase's partition is the
// identity).  Before, every sub-step ran the full formula for every cell: 256^2 1.19 ms a call of 200
// sub-steps, 128^3 8.5 ms.
//
// What a call needs besides the caller's arrays is in file-scope device arrays with room for
// kNoAllocMaxCells cells (28.5 MiB), which every GPU the library is loaded on holds until the process
// ends: Jacobi sub-steps' second concentration buffer (16 MiB), the list of the cells that need the
// full formula (8 MiB), unit-phase bytes, flags and packed flags (4.5 MiB).  Host code never passes an
// array's name to a kernel: the device addresses are looked up once per device with
// hipGetSymbolAddress (with that device current) and kept per device.  No part needs clearing: every
// pass writes what the next one reads.  Calls on one GPU share the arrays, so calls whose work
// overlaps on one GPU (two streams, two threads) race; calls ordered on one stream do not.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>

#include "../../include/phasefield_amd.h"
#include "pf_diffuse_direct.h"
#include "pf_diffuse_tile.h"
#include "pf_handle_access.h"

using namespace pfamd;

namespace {

constexpr long kNoAllocMaxCells = 1L << 21;  // 2,097,152 cells (e.g. 128^3)
constexpr long kMaxListBlocks = kNoAllocMaxCells / (256L * kListChunk);
__device__ __align__(256) double scratch[kNoAllocMaxCells];
__device__ __align__(256) int cell_list[kNoAllocMaxCells];
__device__ __align__(256) uint8_t unit_bytes[kNoAllocMaxCells];
__device__ __align__(256) uint8_t flag_bytes[kNoAllocMaxCells];
__device__ __align__(256) uint32_t packed_flags[kNoAllocMaxCells / 16];
__device__ __align__(256) int list_offsets[kMaxListBlocks + 1];
__device__ unsigned phase_counts[4];

struct Buffers {
  double *conc;
  int *list, *offsets;
  uint8_t *unit, *flag;
  uint32_t *packed;
  unsigned *count;
};

constexpr int kMaxDevices = 64;
std::mutex g_buffers_mutex;
std::array<Buffers, kMaxDevices> g_buffers{};

// device addresses of the arrays on the current device (looked up on the first call there)
hipError_t buffers_on(int dev, Buffers *out) {
  std::lock_guard<std::mutex> lock(g_buffers_mutex);
  Buffers &b = g_buffers[dev];
  if (!b.conc) {
    Buffers n{};
    auto get = [](auto *&ptr, const void *symbol) {
      void *p = nullptr;
      const hipError_t e = hipGetSymbolAddress(&p, symbol);
      ptr = static_cast<std::remove_reference_t<decltype(ptr)>>(p);
      return e;
    };
    hipError_t e = get(n.list, HIP_SYMBOL(cell_list));
    if (e == hipSuccess) e = get(n.offsets, HIP_SYMBOL(list_offsets));
    if (e == hipSuccess) e = get(n.unit, HIP_SYMBOL(unit_bytes));
    if (e == hipSuccess) e = get(n.flag, HIP_SYMBOL(flag_bytes));
    if (e == hipSuccess) e = get(n.packed, HIP_SYMBOL(packed_flags));
    if (e == hipSuccess) e = get(n.count, HIP_SYMBOL(phase_counts));
    if (e == hipSuccess) e = get(n.conc, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    b = n;
  }
  *out = b;
  return hipSuccess;
}

__global__ __launch_bounds__(256) void copy_conc_kernel(const double *__restrict__ src,
                                                        double *__restrict__ dst, long n) {
  const long i = long(blockIdx.x) * 256 + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

}  // namespace

extern "C" int pf_gpu_diffusion_solver_noalloc(const double *hdiffusivity,
                                               const double *hpartition_k,
                                               const double *hpartition_c,
                                               const double *dvalue_phase, double *dtotal_conc,
                                               int x, int y, int z, double dt, double dx,
                                               void *stream) {
  if (!hdiffusivity || !hpartition_k || !hpartition_c || !dvalue_phase || !dtotal_conc)
    return set_global_error(PF_ERR_INVALID, "pf_gpu_diffusion_solver_noalloc: null pointer");
  if (x < 1 || y < 1 || z < 1 || (y == 1 && z == 1))
    return set_global_error(PF_ERR_INVALID,
                            "pf_gpu_diffusion_solver_noalloc: extents must be >= 1 and not 1D");
  const long N = long(x) * y * z;
  if (N > kNoAllocMaxCells)
    return set_global_error(
        PF_ERR_RANGE, "pf_gpu_diffusion_solver_noalloc: " + std::to_string(N) +
                          " cells exceed its scratch buffer of " +
                          std::to_string(kNoAllocMaxCells) + " cells; use pf_gpu_diffusion_solver");
  if (!(dx > 0) || !(dt >= 0))
    return set_global_error(PF_ERR_INVALID, "pf_gpu_diffusion_solver_noalloc: bad dt or dx");
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_global_error(PF_ERR_NODEVICE, "pf_gpu_diffusion_solver_noalloc: no current device");
  Buffers buf;
  if ((e = buffers_on(dev, &buf)) != hipSuccess)
    return set_global_error(PF_ERR_HIP, std::string("pf_gpu_diffusion_solver_noalloc: "
                                                    "hipGetSymbolAddress: ") +
                                            hipGetErrorString(e));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // sub-step count and factor exactly as pf_gpu_diffusion_solver (gpu_solver.cpp:205-209)
  const int dims = z > 1 ? 3 : 2;
  const double max_diff = *std::max_element(hdiffusivity, hdiffusivity + 3);
  const double del_t = dx * dx / max_diff / dims * 0.2f;
  const int num_loop = int(std::ceil(dt / del_t));
  if (num_loop <= 0) return PF_OK;
  DiffConsts<double> dc;
  std::memset(&dc, 0, sizeof(dc));
  for (int i = 0; i < 3; ++i) {
    for (int j = 0; j < 3; ++j) {
      dc.pk[i][j] = hpartition_k[i + 3 * j];  // column-major (i,j) at i+3j
      dc.pc[i][j] = hpartition_c[i + 3 * j];
    }
    dc.D[i] = hdiffusivity[i];
  }
  dc.r = dt / num_loop / (dx * dx);
  const double *pf = dvalue_phase;
  double *a = dtotal_conc, *b = buf.conc;
  // Phases whose bulk cells take the reduced form: identity partition.  None where a constant is not
  // finite: the full formula multiplies it by the zeros of absent phases, which the reduced form drops.
  bool finite = true;
  for (int i = 0; i < 3; ++i) {
    finite = finite && std::isfinite(dc.D[i]);
    for (int j = 0; j < 3; ++j) finite = finite && std::isfinite(dc.pk[i][j]) && std::isfinite(dc.pc[i][j]);
  }
  unsigned mask = 0;
  for (int p = 0; p < 3; ++p)
    if (finite && dc.pk[p][p] == 1.0 && dc.pc[p][p] == 0.0) mask |= 1u << (p + 1);
  TileGeom tile;
  const bool tiles = z == 1 && tile_geometry(x, y, 1, false, num_loop, nullptr, tile);
  // (six faces always, as Diff3D sums them, gpu_solver.cpp:160-188)
  // No phase has a reduced form: every cell takes the full formula, which the LDS-tiled kernel shares
  // between neighbours (128^3, 200 sub-steps: 8.59 ms, 13.71 with every cell listed).  Its columns leave a
  // smaller domain's latency bare (60^3 8.18 ms, 2.88 with every cell listed).
  const bool full = !mask && !tiles && N > (1L << 20);
  if (!full)
    e = launch_classify<double, 3, 6, false>(s, pf, buf.unit, buf.flag, x, y, z, N, mask, buf.count);
  if (e != hipSuccess)
    return set_global_error(PF_ERR_HIP, std::string("pf_gpu_diffusion_solver_noalloc: launch: ") +
                                            hipGetErrorString(e));
  if (tiles) {
    for (int left = num_loop; left > 0; left -= tile.steps) {
      (void)tile_geometry(x, y, 1, false, left, nullptr, tile);
      hipLaunchKernelGGL((diffuse_tile_kernel<FormF64, 3, true>), dim3(unsigned(tile.nblocks)),
                         dim3(kTileNT), 0, s, a, b, pf, buf.flag, dc, tile, N, 0u, 0);
      std::swap(a, b);
    }
  } else if (full) {
    // 64 x kDiffTY columns, z split into chunks of >= 16 planes until about 2048 workgroups.
    const int tiles_x = (x + 63) / 64, tiles_y = (y + kDiffTY - 1) / kDiffTY;
    const long columns = long(tiles_x) * tiles_y;
    const long nzc = std::max(1L, std::min<long>(z, (2048 + columns - 1) / columns));
    const int zc = std::max(int((z + nzc - 1) / nzc), std::min(z, 16));
    const int nblocks = int(columns * ((z + zc - 1) / zc));
    for (int it = 0; it < num_loop; ++it) {
      hipLaunchKernelGGL((diffuse_kernel<FormF64, 3, 6, false, kDiffTY>), dim3(unsigned(nblocks)),
                         dim3(64, kDiffTY + 3), 0, s, a, b, pf, dc, x, y, z, zc, tiles_x, tiles_y, nblocks);
      std::swap(a, b);
    }
  } else {
    const unsigned nl = unsigned((N + 256L * kListChunk - 1) / (256L * kListChunk));
    hipLaunchKernelGGL(general_count_kernel, dim3(nl), dim3(256), 0, s, buf.flag,
                       static_cast<const unsigned *>(nullptr), N, buf.offsets, ListOrder{},
                       static_cast<int *>(nullptr), buf.packed);
    hipLaunchKernelGGL(general_scan_kernel, dim3(1), dim3(1024), 0, s, buf.offsets, int(nl),
                       static_cast<int *>(nullptr));
    hipLaunchKernelGGL(general_scatter_kernel, dim3(nl), dim3(256), 0, s, buf.flag,
                       static_cast<const unsigned *>(nullptr), N, buf.offsets, buf.list, ListOrder{});
    for (int it = 0; it < num_loop && e == hipSuccess; ++it) {
      e = launch_direct<FormF64, 3, false>(s, a, b, pf, buf.packed, buf.list, buf.offsets + nl, dc, x,
                                           y, z, (it & 1) != 0);
      std::swap(a, b);
    }
    if (e != hipSuccess)
      return set_global_error(PF_ERR_HIP, std::string("pf_gpu_diffusion_solver_noalloc: launch: ") +
                                              hipGetErrorString(e));
  }
  if (a != dtotal_conc)  // an odd number of launches leaves the result in the scratch buffer
    hipLaunchKernelGGL(copy_conc_kernel, dim3(unsigned((N + 255) / 256)), dim3(256), 0, s, a,
                       dtotal_conc, N);
  if ((e = hipGetLastError()) != hipSuccess)
    return set_global_error(PF_ERR_HIP, std::string("pf_gpu_diffusion_solver_noalloc: launch: ") +
                                            hipGetErrorString(e));
  return PF_OK;
}
