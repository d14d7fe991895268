// All-pairs execute of the FP32-FFT form that allocates nothing
// (sxc_plan_execute_noalloc, include/seismic_xcorr.h).
//
// No counterpart in the reference.  It serves callers that cannot call
// hipMalloc -- code under HIP graph capture, tight serving loops, harnesses
// that forbid allocation -- and runs the kernels of sxc_plan_execute at the same
// period and on the same segments of the rows, so that the results are the same bit
// for bit.  A job whose rows are cut and whose spectra do not fit runs in pairs of
// event bands.  The workspace (spectra, norms, demeaned
// traces, work list, near-tie records and counter, and the
// twiddle tables of every FFT period) lives in one file-scope device array,
// `scratch`, of kScratchBytes per GPU, held until the process ends.
//
// The array's name is a host-side stand-in in host code: its device address
// is taken once per device with hipGetSymbolAddress (first call on that
// device, with it current) and only that address is used afterwards.  The
// twiddle tables are copied in at that point; the rest is laid out per call.
// Every call on one GPU shares its array, so calls that overlap on one GPU
// (concurrent streams or host threads) race: callers must order them.
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "../../include/seismic_xcorr.h"
#include "xc_engine.h"
#include "xc_kernels.h"
#include "xc_plan.h"

// Workspace of the no-allocation entry point, per GPU.
constexpr size_t kScratchBytes = 128ull << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace sxc {
namespace {

constexpr long long kNoallocTieCap = 1LL << 20;  // near-tie records (16 B each)
constexpr int kMaxDevices = 64;
constexpr int kRadices[] = {8, 16, 24, 32, 40, 48, 64};

// Work items (row i, first column) of column chunk c = blockIdx.x of the columns
// [col0, col0 + n), in the chunk-major order of the plan's host-built list.
// Rows before the columns: every one of them per chunk.  The columns' own
// triangle (row0 == col0): with K columns per chunk, chunk c holds its rows 0 ..
// min(N, K (c + 1)) - 1, and chunks before it min(N, K (c' + 1)) each, i.e. K/2 c
// (c + 1) items while K (c' + 1) <= N, then N per chunk.
__global__ __launch_bounds__(256) void k_fill_work(int2* work, int row0, int rows, int col0, int n, int chunk) {
  const long long c = blockIdx.x;
  const int j0 = (int)(c * chunk);
  if (row0 != col0) {
    for (int i = threadIdx.x; i < rows; i += blockDim.x) work[c * rows + i] = make_int2(row0 + i, col0 + j0);
    return;
  }
  const long long q = n / chunk;  // chunks whose K (c' + 1) <= N
  const long long half = chunk / 2;
  const long long off = c <= q ? half * c * (c + 1) : half * q * (q + 1) + (c - q) * n;
  const int j1 = min(n, j0 + chunk);
  for (int i = threadIdx.x; i < j1; i += blockDim.x) work[off + i] = make_int2(row0 + i, col0 + max(i, j0));
}

struct TableOffsets {
  size_t fwd = 0, inv = 0, post = 0;  // byte offsets into the scratch array
};

struct DeviceScratch {
  unsigned char* base = nullptr;  // device address of `scratch` on this device
  size_t tables_end = 0;          // bytes used by the twiddle tables
  TableOffsets tab[65];           // by R
};

std::mutex g_mu;
DeviceScratch g_dev[kMaxDevices];

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// First call on a device (that device current): the array's address, then
// the twiddle tables of every period copied in.
int scratch_for_device(int dev, DeviceScratch** out) {
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("device %d beyond the %d devices the no-allocation entry point tracks", dev, kMaxDevices);
    return SXC_ERR_INVALID;
  }
  std::lock_guard<std::mutex> lk(g_mu);
  DeviceScratch& ds = g_dev[dev];
  if (ds.base) {
    *out = &ds;
    return SXC_OK;
  }
  void* ptr = nullptr;
  hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    set_error("hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    return SXC_ERR_HIP;
  }
  size_t off = 0;
  DeviceScratch tmp;
  for (int R : kRadices) {
    const int M = 64 * R, P = 2 * M;
    std::vector<float2> fw = wave_tables(R, -1), iw = wave_tables(R, +1), post(M + 1);
    for (int k = 0; k <= M; ++k) twiddle(k, P, -1, &post[k].x, &post[k].y);
    TableOffsets& t = tmp.tab[R];
    t.fwd = off;
    off = align256(off + fw.size() * sizeof(float2));
    t.inv = off;
    off = align256(off + iw.size() * sizeof(float2));
    t.post = off;
    off = align256(off + post.size() * sizeof(float2));
    unsigned char* b = (unsigned char*)ptr;
    if (hipMemcpy(b + t.fwd, fw.data(), fw.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b + t.inv, iw.data(), iw.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(b + t.post, post.data(), post.size() * sizeof(float2), hipMemcpyHostToDevice) != hipSuccess) {
      set_error("copying the twiddle tables into the scratch array failed");
      return SXC_ERR_HIP;
    }
  }
  tmp.tables_end = off;
  tmp.base = (unsigned char*)ptr;
  ds = tmp;
  *out = &ds;
  return SXC_OK;
}

}  // namespace
}  // namespace sxc

using namespace sxc;

namespace {
// Byte offsets of a call's workspace after the tables.
struct Layout {
  size_t norms, traces, ties, count, work, spec, end;
};
Layout layout(const sxc_plan& p, size_t begin, long long n_work, size_t spec_elems) {
  const long long rows = (long long)p.d.n_events * p.d.n_channels;
  Layout l;
  size_t off = begin;
  auto part = [&](size_t bytes) {
    const size_t at = off;
    off = align256(off + bytes);
    return at;
  };
  l.norms = part((size_t)rows * sizeof(double));
  l.traces = part(p.d.demean ? (size_t)rows * p.P * sizeof(float) : 0);
  l.ties = part((size_t)p.tie_cap * sizeof(int4));
  l.count = part(sizeof(unsigned));
  l.work = part((size_t)n_work * sizeof(int2));
  l.spec = part(spec_elems * sizeof(float2));
  l.end = off;
  return l;
}
// Work items of n columns' own triangle, or of as many rows before them: the
// larger of the two.
long long band_items(int n, int chunk) { return (long long)n * ((n + chunk - 1) / chunk); }
}  // namespace

// small: rows kept whole and the longest column chunks.
static int execute_noalloc(const sxc_plan_desc* desc, bool small, const float* d_traces, long long trace_stride,
                           int in_len, float* d_vals_pos, int* d_lags_pos, float* d_vals_neg, int* d_lags_neg,
                           void* stream) {
  int rc;
  sxc_plan p;
  p.chunk = small ? 64 : 0;
  fft_plan_geometry(*desc, kNoallocTieCap, small ? Rows::kWhole : Rows::kCut, &p);
  if (in_len < 1 || in_len > p.P || trace_stride < in_len) {
    set_error("in_len %d must be in [1, P=%d] and <= trace_stride %lld", in_len, p.P, trace_stride);
    return SXC_ERR_INVALID;
  }
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    set_error("no HIP device");
    return SXC_ERR_HIP;
  }
  DeviceScratch* ds = nullptr;
  if ((rc = scratch_for_device(dev, &ds))) return rc;
  Layout l = layout(p, ds->tables_end, p.n_work, p.spec_elems);
  int band = 0;  // events of a band, 0: the whole job at once
  if (l.end > kScratchBytes && !small) {
    // a job at the limit keeps the fewest spectra and the shortest work list; where
    // a plan's execute cuts these rows, so do the bands
    sxc_plan whole;
    whole.chunk = 64;
    fft_plan_geometry(*desc, kNoallocTieCap, Rows::kWhole, &whole);
    const bool fits = layout(whole, ds->tables_end, whole.n_work, whole.spec_elems).end <= kScratchBytes;
    const int n_seg = fft_geom(&p, in_len, false).n_seg;
    if (!fits || !n_seg)
      return execute_noalloc(desc, true, d_traces, trace_stride, in_len, d_vals_pos, d_lags_pos, d_vals_neg,
                             d_lags_neg, stream);
    const size_t event_elems = (size_t)desc->n_channels * n_seg * p.cut.spec_stride;
    for (int k = 2; l.end > kScratchBytes && band != p.chunk; ++k) {
      band = ((desc->n_events + k - 1) / k + p.chunk - 1) / p.chunk * p.chunk;
      l = layout(p, ds->tables_end, band_items(band, p.chunk), 2 * band * event_elems);
    }
  }
  if (l.end > kScratchBytes) {
    set_error("this job needs %zu bytes of workspace; the no-allocation entry point holds at most %zu "
              "(%zu after the twiddle tables): use sxc_plan_execute",
              l.end, kScratchBytes, kScratchBytes - ds->tables_end);
    return SXC_ERR_INVALID;
  }
  unsigned char* b = ds->base;
  p.spec = (float2*)(b + l.spec);
  p.norms = (double*)(b + l.norms);
  p.traces = desc->demean ? (float*)(b + l.traces) : nullptr;
  p.work = (int2*)(b + l.work);
  p.ties = (int4*)(b + l.ties);
  p.tie_count = (unsigned*)(b + l.count);
  p.fwd2 = (float2*)(b + ds->tab[p.R].fwd);
  p.inv2 = (float2*)(b + ds->tab[p.R].inv);
  p.post = (float2*)(b + ds->tab[p.R].post);
  for (FftGeom* g : {&p.narrow, &p.cut})
    if (g->P) {
      g->fwd2 = (float2*)(b + ds->tab[g->R].fwd);
      g->inv2 = (float2*)(b + ds->tab[g->R].inv);
      g->post = (float2*)(b + ds->tab[g->R].post);
    }
  p.device = dev;
  hipStream_t st = (hipStream_t)stream;
  p.last_stream = st;
  // the work list of these rows and columns (the previous call's contents are
  // stale); the tie counter is cleared by the execute itself
  auto fill = [&](int row0, int rows, int col0, int cols) -> int {
    const int n_chunks = (cols + p.chunk - 1) / p.chunk;
    hipLaunchKernelGGL(k_fill_work, dim3(n_chunks), dim3(256), 0, st, p.work, row0, rows, col0, cols, p.chunk);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      set_error("scratch set-up launches failed: %s", hipGetErrorString(e));
      return SXC_ERR_HIP;
    }
    return (int)(row0 == col0 ? triangle_items(cols, p.chunk) : (long long)rows * n_chunks);
  };
  if (band) {
    const FftGeom g = fft_geom(&p, in_len, false);
    float2* cols = p.spec + (size_t)band * desc->n_channels * g.n_seg * g.spec_stride;
    return fft_plan_execute_bands(&p, g, band, p.spec, cols, d_traces, trace_stride, in_len, d_vals_pos, d_lags_pos,
                                  d_vals_neg, d_lags_neg, fill, st);
  }
  const int n_work = fill(0, desc->n_events, 0, desc->n_events);
  if (n_work < 0) return n_work;
  return fft_plan_execute(&p, d_traces, nullptr, trace_stride, in_len, d_vals_pos, d_lags_pos, d_vals_neg,
                          d_lags_neg, st);
}

extern "C" int sxc_plan_execute_noalloc(const sxc_plan_desc* desc, const float* d_traces, long long trace_stride,
                                        int in_len, float* d_vals_pos, int* d_lags_pos, float* d_vals_neg,
                                        int* d_lags_neg, void* stream) {
  clear_error();
  if (!desc || !d_traces || !d_vals_pos || !d_lags_pos || !d_vals_neg || !d_lags_neg) {
    set_error("null argument");
    return SXC_ERR_INVALID;
  }
  int rc = validate_desc(*desc);
  if (rc) return rc;
  if (desc->form != SXC_FORM_FFT_F32) {
    set_error("the no-allocation entry point runs the FFT form only");
    return SXC_ERR_INVALID;
  }
  return execute_noalloc(desc, false, d_traces, trace_stride, in_len, d_vals_pos, d_lags_pos, d_vals_neg, d_lags_neg,
                         stream);
}
