// Stateless C entry points: errors, device query, SDF and sizing evaluation,
// 3D quality kernels and gradient limiting.
#include <cstdarg>
#include <cstdio>
#include <cstring>

#include "common.h"
#include "sdf_eval.h"
#include "quality3d.h"
#include "sizing_eval.h"

static thread_local char g_err[512] = "";

int sm_set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

extern "C" int sm_version(void) { return 100; }

extern "C" int sm_last_error(char *buf, size_t len) {
  if (!buf || len == 0) return SM_ERR_ARG;
  std::strncpy(buf, g_err, len - 1);
  buf[len - 1] = 0;
  return SM_OK;
}

extern "C" int sm_device_count(int *count) {
  if (!count) return SM_ERR_ARG;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) n = 0;
  int usable = 0;
  for (int d = 0; d < n; ++d) {
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, d) != hipSuccess) continue;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) == 0) ++usable;
  }
  *count = usable;
  return SM_OK;
}

namespace {

using namespace smk;

template <int DIM>
__global__ void k_sdf(const sm_node *tape, int ntape, const double *x, int64_t n, double *d) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double q[3];
#pragma unroll
  for (int k = 0; k < DIM; ++k) q[k] = x[i * DIM + k];
  d[i] = sdf_eval<DIM>(tape, ntape, q);
}

template <int DIM>
__global__ void k_sizing(GridView g, const double *x, int64_t n, float *h) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double q[3];
#pragma unroll
  for (int k = 0; k < DIM; ++k) q[k] = x[i * DIM + k];
  h[i] = (float)grid_eval<DIM>(g, q);
}

__global__ void k_dihedral(const double *p, const int32_t *cells, int64_t nc, double *out) {
  int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nc) return;
  int32_t v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = cells[4 * c + k];
#pragma unroll
  for (int i = 0; i < 6; ++i) out[6 * c + i] = dihedral_angle(p, v, i);
}

__global__ void k_circumgrad(const double *q1, const double *q2, const double *q3,
                             const double *q4, int64_t k, double *g) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= k) return;
  circumsphere_grad(q1 + 3 * i, q2 + 3 * i, q3 + 3 * i, q4 + 3 * i, g + 3 * i);
}

// Gradient limiting: the fixed point of FastHJ.cpp's relaxation
// f_i <= f_j + elen*dfdx over the 4/6-neighbour grid stencil is the
// distance transform min_j (f0_j + elen*dfdx * |i - j|_1), which separates
// into a forward and a backward sweep along each grid line of each axis:
// g_j = min(f_j, g_{j-1} + step), rounded step by step.
//
// A sweep is a chain, but a short one in effect: once g_j = f_j the past no
// longer matters, and with l_j the same sweep started at j0 instead of 0,
// g <= l and g_j = l_j from the first equality on (the rounded addition is
// monotone), bit for bit.  So a line is cut into segments swept side by
// side in LDS, and each segment then takes the value carried in from the one
// before until it meets what is there already; that is repeated while the
// last value of some segment changes (a limited slope across k segments
// takes k rounds).  Bound: HBM, one read and one write of
// the grid per axis (one thread a line, as before, left the chip with the
// 5395 lines of a 2D model: 21 workgroups, a dependent global access per
// value and sweep).  Measured on MI355X, 1911 x 5395, with the copy of the
// grid its caller makes: 4.91 ms before, 0.37 now.
constexpr int kLimSeg = 16;     // values a thread sweeps
constexpr int kLimMax = 16384;  // longest line held in LDS (128 KiB)
// values a workgroup holds: of rows (with one of padding each; half a CU's
// LDS) and of columns, or one line, and the dynamic LDS that takes at most
constexpr int kLimRows = 9216, kLimColumns = 18432;
constexpr int kLimRowsLds = (kLimMax + 1) * (int)sizeof(double);
constexpr int kLimColumnsLds = kLimColumns * (int)sizeof(double);

// The sweeps of `lines` lines of `len` values held in LDS with stride `ls`
// (line l at l * ll): every thread of the workgroup takes segments.
__device__ inline void limit_lines(double *sh, int lines, int len, int ls, int ll, double step,
                                   int *changed) {
  const int segs = (len + kLimSeg - 1) / kLimSeg;
  const auto at = [&](int l, int j) -> double & { return sh[l * ll + j * ls]; };
  for (int dir = 0; dir < 2; ++dir) {
    __syncthreads();
    // each segment on its own
    for (int w = threadIdx.x; w < lines * segs; w += blockDim.x) {
      const int l = w % lines, sg = w / lines;
      const int j0 = sg * kLimSeg, n = min(kLimSeg, len - j0);
      double prev = 0.0;
      for (int i = 0; i < n; ++i) {
        double &v = at(l, dir == 0 ? j0 + i : j0 + n - 1 - i);
        const double lim = prev + step;
        if (i > 0 && v > lim) v = lim;
        prev = v;
      }
    }
    // then what each carries into the next, until nothing changes.  The last
    // value of a segment is read by the next one's thread while its own may
    // lower it: a relaxed atomic, the old value or the new one (after the old
    // one another round follows).  Reading all of them before a further
    // barrier took 4 % longer.
    const auto read = [&](int l, int j) {
      return __hip_atomic_load(&at(l, j), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    for (;;) {
      __syncthreads();
      if (threadIdx.x == 0) *changed = 0;
      __syncthreads();
      for (int w = threadIdx.x; w < lines * (segs - 1); w += blockDim.x) {
        const int l = w % lines, q = 1 + w / lines;
        int j = dir == 0 ? q * kLimSeg : (segs - q) * kLimSeg - 1;
        const int end = dir == 0 ? min(len, j + kLimSeg) : j - kLimSeg;
        const int inc = dir == 0 ? 1 : -1;
        double prev = read(l, j - inc);
        for (int i = 0; j != end; j += inc, ++i) {
          const double lim = prev + step;
          if (!(read(l, j) > lim)) break;
          __hip_atomic_store(&at(l, j), lim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          prev = lim;
          if (i == kLimSeg - 1 || j + inc == end) *changed = 1;
        }
      }
      __syncthreads();
      if (*changed == 0) break;
    }
  }
  __syncthreads();
}

// Lines contiguous in memory (axis 0): whole lines per workgroup.
__global__ __launch_bounds__(256) void k_limgrad_rows(double *f, int len, int64_t lines, int per,
                                                      double step) {
  extern __shared__ double sh[];
  __shared__ int changed;
  const int64_t l0 = (int64_t)blockIdx.x * per;
  const int nl = (int)(lines - l0 < per ? lines - l0 : per);
  double *p = f + l0 * len;
  // one word of padding a line keeps the lines' values off one bank
  for (int l = 0; l < nl; ++l)
    for (int j = threadIdx.x; j < len; j += blockDim.x) sh[l * (len + 1) + j] = p[(int64_t)l * len + j];
  limit_lines(sh, nl, len, 1, len + 1, step, &changed);
  for (int l = 0; l < nl; ++l)
    for (int j = threadIdx.x; j < len; j += blockDim.x) p[(int64_t)l * len + j] = sh[l * (len + 1) + j];
}

// Lines of stride `stride`, neighbours in memory: `per` of them a workgroup.
__global__ __launch_bounds__(256) void k_limgrad_columns(double *f, int len, int64_t stride,
                                                         int64_t outer, int per, double step) {
  extern __shared__ double sh[];
  __shared__ int changed;
  const int64_t c0 = (int64_t)xcd_block() * per;
  const int nc = (int)(stride - c0 < per ? stride - c0 : per);
  double *p = f + (int64_t)blockIdx.y * outer + c0;
  for (int e = threadIdx.x; e < len * per; e += blockDim.x) {
    const int j = e / per, c = e % per;
    if (c < nc) sh[e] = p[(int64_t)j * stride + c];
  }
  limit_lines(sh, nc, len, per, 1, step, &changed);
  for (int e = threadIdx.x; e < len * per; e += blockDim.x) {
    const int j = e / per, c = e % per;
    if (c < nc) p[(int64_t)j * stride + c] = sh[e];
  }
}

// Lines longer than LDS holds, and short rows: one thread a line.
__global__ void k_limgrad_axis(double *f, int64_t lines, int64_t len, int64_t stride,
                               int64_t outer, double step) {
  const int64_t line = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (line >= lines) return;
  const int64_t base = (line / stride) * outer + line % stride;
  double prev = f[base];
  for (int64_t j = 1; j < len; ++j) {
    double cur = f[base + j * stride];
    double lim = prev + step;
    if (cur > lim) cur = lim;
    f[base + j * stride] = cur;
    prev = cur;
  }
  prev = f[base + (len - 1) * stride];
  for (int64_t j = len - 2; j >= 0; --j) {
    double cur = f[base + j * stride];
    double lim = prev + step;
    if (cur > lim) cur = lim;
    f[base + j * stride] = cur;
    prev = cur;
  }
}

}  // namespace

extern "C" int sm_sdf_eval(const sm_node *tape, int ntape, int dim, const double *x, int64_t n,
                           double *d, void *stream) {
  SM_CHECK(dim == 2 || dim == 3, SM_ERR_ARG, "sdf_eval: dim must be 2 or 3");
  SM_CHECK(n >= 0 && ntape > 0, SM_ERR_ARG, "sdf_eval: bad size");
  if (n == 0) return SM_OK;
  SM_CHECK(tape && x && d, SM_ERR_ARG, "sdf_eval: null pointer");
  hipStream_t s = stream_of(stream);
  if (dim == 2)
    hipLaunchKernelGGL(k_sdf<2>, dim3(blocks_for(n, 256)), dim3(256), 0, s, tape, ntape, x, n, d);
  else
    hipLaunchKernelGGL(k_sdf<3>, dim3(blocks_for(n, 256)), dim3(256), 0, s, tape, ntape, x, n, d);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int sm_sizing_eval(const sm_grid *grid, const double *x, int64_t n, float *h,
                              void *stream) {
  SM_CHECK(grid && (grid->dim == 2 || grid->dim == 3), SM_ERR_ARG, "sizing_eval: bad grid");
  SM_CHECK(n >= 0, SM_ERR_ARG, "sizing_eval: bad size");
  if (n == 0) return SM_OK;
  SM_CHECK(x && h, SM_ERR_ARG, "sizing_eval: null pointer");
  GridView g{};
  g.dim = grid->dim;
  g.values = grid->values;
  g.hconst = grid->hconst;
  for (int k = 0; k < 3; ++k) {
    g.n[k] = grid->n[k];
    g.axis[k] = grid->axis[k];
  }
  if (g.values)
    for (int k = 0; k < g.dim; ++k)
      SM_CHECK(g.n[k] >= 2 && g.axis[k], SM_ERR_ARG, "sizing_eval: axis %d invalid", k);
  hipStream_t s = stream_of(stream);
  if (g.dim == 2)
    hipLaunchKernelGGL(k_sizing<2>, dim3(blocks_for(n, 256)), dim3(256), 0, s, g, x, n, h);
  else
    hipLaunchKernelGGL(k_sizing<3>, dim3(blocks_for(n, 256)), dim3(256), 0, s, g, x, n, h);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int sm_dihedral_angles(const double *p, const int32_t *cells, int64_t ncells,
                                  double *angles, void *stream) {
  SM_CHECK(ncells >= 0, SM_ERR_ARG, "dihedral_angles: bad size");
  if (ncells == 0) return SM_OK;
  SM_CHECK(p && cells && angles, SM_ERR_ARG, "dihedral_angles: null pointer");
  hipLaunchKernelGGL(k_dihedral, dim3(blocks_for(ncells, 256)), dim3(256), 0, stream_of(stream),
                     p, cells, ncells, angles);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int sm_circumsphere_grad(const double *p0, const double *p1, const double *p2,
                                    const double *p3, int64_t k, double *grad, void *stream) {
  SM_CHECK(k >= 0, SM_ERR_ARG, "circumsphere_grad: bad size");
  if (k == 0) return SM_OK;
  SM_CHECK(p0 && p1 && p2 && p3 && grad, SM_ERR_ARG, "circumsphere_grad: null pointer");
  hipLaunchKernelGGL(k_circumgrad, dim3(blocks_for(k, 256)), dim3(256), 0, stream_of(stream),
                     p0, p1, p2, p3, k, grad);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int sm_limgrad(double *f, int nz, int nx, int ny, double elen, double dfdx,
                          void *stream) {
  SM_CHECK(f && nz > 0 && nx > 0 && ny > 0, SM_ERR_ARG, "limgrad: bad argument");
  const double step = elen * dfdx;
  hipStream_t s = stream_of(stream);
  const int dims[3] = {nz, nx, ny};
  int64_t stride = 1;
  for (int axis = 0; axis < 3; ++axis) {
    const int len = dims[axis];
    const int64_t lines = (int64_t)nz * nx * ny / len, outer = stride * len;
    if (len >= 2) {
      // One thread a line: lines longer than LDS holds, more planes than
      // grid.y counts (columns only: rows have none), and short rows.  Of
      // those a thread's cache lines serve all of its few steps, and a
      // workgroup of the rows kernel has little to sweep: 1000 lines of 20
      // values 34 against 56 us for all three axes of the grid, 60000 of 16
      // 57 against 69, 457 k of 8 172 against 224; but 457 k of 12 279
      // against 258 and 457 k of 210 8.9 against 4.1 ms.
      const bool few = stride == 1 && (len <= 10 || (len <= 64 && lines * len <= 1 << 21));
      // rows: as many lines as fill half a CU's LDS (two workgroups then
      // hide each other's loads), at least one; columns: a power of two of
      // them (64-byte runs at 8), fewer when the lines are long
      if (len > kLimMax || (stride > 1 && lines / stride > 65535) || few) {
        hipLaunchKernelGGL(k_limgrad_axis, dim3(blocks_for(lines, 64)), dim3(64), 0, s, f, lines,
                           len, stride, outer, step);
      } else if (stride == 1) {
        int per = kLimRows / (len + 1);
        per = per < 1 ? 1 : (per > 64 ? 64 : per);
        const size_t lds = (size_t)per * (len + 1) * sizeof(double);
        // the kernel's own bound, the same for every call: a call's own size
        // could be another thread's too little
        SM_HIP(hipFuncSetAttribute((const void *)k_limgrad_rows,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kLimRowsLds));
        hipLaunchKernelGGL(k_limgrad_rows, dim3((unsigned)((lines + per - 1) / per)), dim3(256),
                           lds, s, f, len, lines, per, step);
      } else {
        int per = 64;
        while (per > 1 && (int64_t)per * len > kLimColumns) per /= 2;
        while (per > 8 && (stride + per - 1) / per * (lines / stride) < 512) per /= 2;
        const size_t lds = (size_t)per * len * sizeof(double);
        SM_HIP(hipFuncSetAttribute((const void *)k_limgrad_columns,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kLimColumnsLds));
        hipLaunchKernelGGL(k_limgrad_columns,
                           dim3((unsigned)((stride + per - 1) / per), (unsigned)(lines / stride)),
                           dim3(256), lds, s, f, len, stride, outer, per, step);
      }
      SM_LAUNCH_CHECK();
    }
    stride = outer;
  }
  return SM_OK;
}
