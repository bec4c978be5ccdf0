// rq_api.cpp -- the C ABI of librq (include/rq.h): argument checks, handle
// ownership, device binding and dispatch to the HIP kernels.
//
// Error rules follow the reference: dequant_tensor's Unsupported / Overflow /
// Truncated (crates/runtimed-gguf/src/quant/dequant.rs:84-95) for block
// streams, ModelError::Shape for activation shapes (linear_layer.rs:88-94).
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <string>
#include <vector>

#include "rq_internal.h"

namespace rq {

static thread_local std::string g_last_error;

int set_error(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return code;
}

hipStream_t as_stream(void *s) { return static_cast<hipStream_t>(s); }

void clear_error() { g_last_error.clear(); }

int fp8_gemm_checks(int xtype, int64_t m, int64_t n, int64_t k, int ytype, int mode) {
  clear_error();
  if (xtype != RQ_F8E4M3 && xtype != RQ_F32 && xtype != RQ_F16 && xtype != RQ_BF16)
    return set_error(RQ_E_ARG, "activation type %d not supported", xtype);
  if (ytype != RQ_F32 && ytype != RQ_F16 && ytype != RQ_BF16)
    return set_error(RQ_E_ARG, "output type %d not supported", ytype);
  if (xtype != RQ_F8E4M3 && mode != RQ_FP8_UNSCALED && mode != RQ_FP8_PER_TOKEN)
    return set_error(RQ_E_ARG, "bad fp8 mode %d", mode);
  if (m < 0 || n <= 0 || k <= 0)
    return set_error(RQ_E_SHAPE, "bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
  return RQ_OK;
}

bool geometry(int qtype, Geometry *g) {
  switch (qtype) {
    case RQ_Q4_0: *g = {32, 18}; return true;
    case RQ_Q5_0: *g = {32, 22}; return true;
    case RQ_Q8_0: *g = {32, 34}; return true;
    case RQ_Q4_K: *g = {256, 144}; return true;
    case RQ_Q5_K: *g = {256, 176}; return true;
    case RQ_Q6_K: *g = {256, 210}; return true;
    default: return false;
  }
}

static bool valid_ftype(int t) { return t == RQ_F32 || t == RQ_F16 || t == RQ_BF16; }

static int hip_check(hipError_t e, const char *what) {
  if (e == hipSuccess) return RQ_OK;
  return set_error(e == hipErrorOutOfMemory ? RQ_E_NOMEM : RQ_E_DEVICE, "%s: %s", what,
                   hipGetErrorString(e));
}

// Dequant_tensor's checks on a flat stream of n_elements (dequant.rs:83-95).
static int stream_checks(int qtype, uint64_t nbytes, uint64_t n_elements, Geometry *g) {
  if (!geometry(qtype, g)) return set_error(RQ_E_UNSUPPORTED, "decode of qtype %d not implemented", qtype);
  if (n_elements % (uint64_t)g->elems != 0)
    return set_error(RQ_E_OVERFLOW, "%llu not a multiple of %d", (unsigned long long)n_elements, g->elems);
  const uint64_t need = n_elements / (uint64_t)g->elems * (uint64_t)g->bytes;
  if (nbytes < need)
    return set_error(RQ_E_TRUNCATED, "truncated: %llu bytes, need %llu", (unsigned long long)nbytes,
                     (unsigned long long)need);
  return RQ_OK;
}

static uint64_t align256(uint64_t v) { return (v + 255) & ~(uint64_t)255; }

// Device bytes of the split layout (rq_internal.h) for nblocks blocks, and
// the offset of its scale array.
static uint64_t split_size(int qtype, uint64_t nblocks, uint64_t *aux_off) {
  const uint64_t qbytes = qtype == RQ_Q8_0 ? 32 : qtype == RQ_Q6_K ? 208 : 16;
  const uint64_t abytes = qtype == RQ_Q5_0 ? 8 : 2;
  *aux_off = align256(nblocks * qbytes);
  return *aux_off + nblocks * abytes;
}

// Host-side split of Q8_0 / Q6_K streams into the aligned device layout
// described in rq_internal.h (small tensors; large ones split on the device).
static void split_layout(int qtype, const uint8_t *src, uint64_t nblocks, std::vector<uint8_t> &dst,
                         uint64_t &aux_off) {
  if (qtype == RQ_Q8_0) {
    aux_off = align256(nblocks * 32);
    dst.assign(aux_off + nblocks * 2, 0);
    for (uint64_t b = 0; b < nblocks; ++b) {
      const uint8_t *blk = src + b * 34;
      memcpy(&dst[b * 32], blk + 2, 32);
      memcpy(&dst[aux_off + b * 2], blk, 2);
    }
  } else if (qtype == RQ_Q4_0) {
    aux_off = align256(nblocks * 16);
    dst.assign(aux_off + nblocks * 2, 0);
    for (uint64_t b = 0; b < nblocks; ++b) {
      const uint8_t *blk = src + b * 18;
      memcpy(&dst[b * 16], blk + 2, 16);
      memcpy(&dst[aux_off + b * 2], blk, 2);
    }
  } else if (qtype == RQ_Q5_0) {
    aux_off = align256(nblocks * 16);
    dst.assign(aux_off + nblocks * 8, 0);
    for (uint64_t b = 0; b < nblocks; ++b) {
      const uint8_t *blk = src + b * 22;
      memcpy(&dst[b * 16], blk + 6, 16);
      memcpy(&dst[aux_off + b * 8], blk + 2, 4);  // qh
      memcpy(&dst[aux_off + b * 8 + 4], blk, 2);  // d
    }
  } else {  // Q6_K
    aux_off = align256(nblocks * 208);
    dst.assign(aux_off + nblocks * 2, 0);
    for (uint64_t b = 0; b < nblocks; ++b) {
      const uint8_t *blk = src + b * 210;
      memcpy(&dst[b * 208], blk, 208);
      memcpy(&dst[aux_off + b * 2], blk + 208, 2);
    }
  }
}

}  // namespace rq

using namespace rq;

extern "C" {

int rq_abi_version(void) { return RQ_ABI_VERSION; }

const char *rq_last_error(void) { return g_last_error.c_str(); }

int rq_weight_create(int qtype, const void *host_blocks, size_t nbytes, int64_t n, int64_t k,
                     int device, rq_weight **out) {
  g_last_error.clear();
  if (!out) return set_error(RQ_E_ARG, "out is null");
  *out = nullptr;
  if (!host_blocks) return set_error(RQ_E_ARG, "host_blocks is null");
  if (n <= 0 || k <= 0) return set_error(RQ_E_SHAPE, "shape [%lld, %lld] must be positive", (long long)n, (long long)k);
  Geometry g;
  const uint64_t count = (uint64_t)n * (uint64_t)k;
  int rc = stream_checks(qtype, nbytes, count, &g);
  if (rc) return rc;
  rc = hip_check(hipSetDevice(device), "hipSetDevice");
  if (rc) return rc;
  const uint64_t nblocks = count / (uint64_t)g.elems;
  const uint8_t *src = static_cast<const uint8_t *>(host_blocks);
  const bool split = qtype == RQ_Q8_0 || qtype == RQ_Q6_K || qtype == RQ_Q4_0 || qtype == RQ_Q5_0;
  const uint64_t raw_bytes = nblocks * (uint64_t)g.bytes;
  uint64_t aux_off = 0, bytes = raw_bytes;
  uint8_t *dptr = nullptr;
  if (raw_bytes >= (4ull << 20)) {
    // Large tensors: pinned double-buffered DMA, split on the device.
    if (split) bytes = split_size(qtype, nblocks, &aux_off);
    rc = hip_check(hipMalloc(reinterpret_cast<void **>(&dptr), bytes), "hipMalloc");
    if (rc) return rc;
    if (split) rc = hip_check(hipMemset(dptr, 0, bytes), "hipMemset");
    if (!rc) rc = upload_blocks(qtype, src, nblocks, g.bytes, dptr, aux_off, device);
  } else {
    std::vector<uint8_t> staged;
    if (split) {
      split_layout(qtype, src, nblocks, staged, aux_off);
      src = staged.data();
      bytes = staged.size();
    }
    rc = hip_check(hipMalloc(reinterpret_cast<void **>(&dptr), bytes), "hipMalloc");
    if (rc) return rc;
    rc = hip_check(hipMemcpy(dptr, src, bytes, hipMemcpyHostToDevice), "hipMemcpy");
  }
  if (rc) {
    (void)hipFree(dptr);
    return rc;
  }
  rq_weight *w = new rq_weight;
  w->qtype = qtype;
  w->device = device;
  w->n = n;
  w->k = k;
  w->gguf_bytes = nblocks * (uint64_t)g.bytes;
  w->nblocks = nblocks;
  w->data = dptr;
  w->data_bytes = bytes;
  w->aux_off = aux_off;
  *out = w;
  return RQ_OK;
}

void rq_weight_destroy(rq_weight *w) {
  if (!w) return;
  int cur = 0;
  if (hipGetDevice(&cur) == hipSuccess && cur != w->device) (void)hipSetDevice(w->device);
  (void)hipFree(w->data);
  if (cur != w->device) (void)hipSetDevice(cur);
  delete w;
}

int rq_weight_info(const rq_weight *w, rq_weight_desc *out) {
  if (!w || !out) return set_error(RQ_E_ARG, "null argument");
  out->qtype = w->qtype;
  out->device = w->device;
  out->n = w->n;
  out->k = w->k;
  out->gguf_bytes = w->gguf_bytes;
  out->device_bytes = w->data_bytes;
  return RQ_OK;
}

int rq_dequant_f32(const rq_weight *w, float *dev_out, void *stream) {
  g_last_error.clear();
  if (!w || !dev_out) return set_error(RQ_E_ARG, "null argument");
  int rc = hip_check(hipSetDevice(w->device), "hipSetDevice");
  if (rc) return rc;
  return launch_dequant_weight(w, dev_out, as_stream(stream));
}

int rq_embedding(const rq_weight *w, const uint32_t *ids, int64_t n_ids, float *dev_out, void *stream) {
  g_last_error.clear();
  if (!w) return set_error(RQ_E_ARG, "weight is null");
  if (n_ids < 0) return set_error(RQ_E_ARG, "n_ids %lld is negative", (long long)n_ids);
  if (n_ids == 0) return RQ_OK;
  if (!ids || !dev_out) return set_error(RQ_E_ARG, "null argument");
  if (w->k % 4 != 0) return set_error(RQ_E_UNSUPPORTED, "row length %lld is not a multiple of 4", (long long)w->k);
  for (int64_t i = 0; i < n_ids; ++i)
    if ((int64_t)ids[i] >= w->n)
      return set_error(RQ_E_ARG, "id %u at position %lld is out of range for %lld rows", ids[i], (long long)i,
                       (long long)w->n);
  int rc = hip_check(hipSetDevice(w->device), "hipSetDevice");
  if (rc) return rc;
  const hipStream_t s = as_stream(stream);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return set_error(RQ_E_ARG, "rq_embedding reads host ids and cannot be captured into a graph");
  }
  rc = launch_gather_args(w, ids, n_ids, dev_out, s);
  if (rc != RQ_E_UNSUPPORTED) return rc;
  WsLease ws(w->device, s);
  uint32_t *dids = static_cast<uint32_t *>(ws.get((size_t)n_ids * sizeof(uint32_t), &rc));
  if (!dids) return rc;
  // From pageable memory the copy returns once the ids are staged, so the
  // caller's buffer may be reused on return.
  rc = hip_check(hipMemcpyAsync(dids, ids, (size_t)n_ids * sizeof(uint32_t), hipMemcpyHostToDevice, s),
                 "hipMemcpyAsync");
  if (!rc) rc = launch_gather_rows(w, dids, n_ids, dev_out, s);
  return rc;
}

int rq_dequant_tensor(int qtype, const void *dev_bytes, size_t nbytes, size_t n_elements,
                      float *dev_out, void *stream) {
  g_last_error.clear();
  Geometry g;
  int rc = stream_checks(qtype, nbytes, n_elements, &g);
  if (rc) return rc;
  if (n_elements == 0) return RQ_OK;
  if (!dev_bytes || !dev_out) return set_error(RQ_E_ARG, "null argument");
  return launch_dequant_raw(qtype, static_cast<const uint8_t *>(dev_bytes),
                            n_elements / (uint64_t)g.elems, dev_out, as_stream(stream));
}

static size_t ftype_bytes(int t) { return t == RQ_F32 ? 4 : 2; }

// Argument checks shared by the linear entry points (linear_layer.rs:88-96
// for the width rule).
static int linear_checks(const rq_weight *w, int xtype, int64_t m, int64_t k, const void *bias, int btype,
                         int ytype) {
  if (!w) return set_error(RQ_E_ARG, "weight is null");
  if (!valid_ftype(xtype)) return set_error(RQ_E_ARG, "activation type %d not supported", xtype);
  if (!valid_ftype(ytype)) return set_error(RQ_E_ARG, "output type %d not supported", ytype);
  if (bias && !valid_ftype(btype)) return set_error(RQ_E_ARG, "bias type %d not supported", btype);
  if (k != w->k)
    return set_error(RQ_E_SHAPE, "linear: expected last dim %lld, got %lld", (long long)w->k, (long long)k);
  if (m < 0) return set_error(RQ_E_SHAPE, "negative row count %lld", (long long)m);
  return RQ_OK;
}

// x as the fused kernels read it: 16-byte aligned, else an aligned copy of
// its m * k elements in the workspace.
static const void *aligned_x(const void *x, int xtype, int64_t m, int64_t k, hipStream_t s, WsLease &ws, int *rc) {
  if (reinterpret_cast<uintptr_t>(x) % 16 == 0) return x;
  const size_t bytes = (size_t)m * (size_t)k * ftype_bytes(xtype);
  void *p = ws.get(bytes, rc);
  if (!p) return nullptr;
  *rc = hip_check(hipMemcpyAsync(p, x, bytes, hipMemcpyDeviceToDevice, s), "hipMemcpyAsync");
  return *rc ? nullptr : p;
}

// Whether a call goes to the codes GEMM, which packs the
// activations in a launch of its own (4-8 us) and reads them in one launch for
// all weights, or to the tiled kernels.  Graph-timed, codes GEMM against
// tiled, us:
//   f32 activations, one weight: 2048 x 2048 at m = 65 / 512 18.3 / 28.2
//     against 24.8 / 29.8 (Q4_K), 17.5 / 26.5 against 28.6 / 33.8 (Q8_0), 8192 x
//     2048 23.9 / 67.9 against 28.7 / 73.6, 2048 x 8192 30.9 / 66.0 against
//     62.2 / 79.5; f16 16.0 / 22.2 against 24.0 / 28.4, 51.6 against 69.8.  The
//     pack does not pay on short rows: 896 x 896 at m = 512 19.3 against 21.7 on
//     the K formats but 17.9 against 16.1 on Q8_0, 1152 x 384 16.7 against 11.6.
//   Sets of weights (q/k/v, gate/up) save a launch a weight and pay throughout.
//   bf16 activations: the tiled kernels round the weights to bf16 as well
//     and take one matrix pass, so only sets on few tiles (m = 333: q/k/v 2048
//     + 2 x 512 rows 29 against 50 us, m = 512: 2 x 2048 rows 35 against 32)
//     and long rows on few tiles (896 x 4864 at m = 65 / 512 22 / 30 against 29
//     / 32, 4096 x 4096 at m = 65 23.5 against 26.7, 2048 x 2048 16.6 against
//     13.9, 8192 x 2048 at m = 512 54 against 33) pay.
// At most 64 rows (32 x 64 tiles up to 32): the small-M kernels read the
// weights a lane its own row, which the vector cache serves one access a lane;
// the codes GEMM reads them coalesced but pays the pack, so it takes the calls
// with many weights.  f32 rows, small-M (m = 2, 3: VALU) against codes, us:
//   m = 5 / 24: Q6_K 2048 x 8192 36.3 / 53.6 against 20.3 / 21.0, 4096 x 14336
//     104 / 135 against 37 / 37, Q4_K 2 x 8192 x 2048 17.3 / 26.2 against 16.7 /
//     17.3, 2 x 14336 x 4096 57 / 91 against 38 / 40, 4096 x 4096 16.6 / 25.4
//     against 16.1 / 16.7, Q8_0 2 x 8192 x 2048 23.9 / 33.7 against 17.0 / 17.7;
//     2 x 2048 x 2048 9.9 / 14.6 against 12.6 / 13.1, 2048 x 2048 6.7 / 8.8
//     against 12.5 / 12.9
//   m = 48 (64 x 64 tiles): 2 x 2048 x 2048 23.5 against 17.9, 2 x 8192 x 2048
//     45.7 against 24.4, Q6_K 2048 x 8192 67.5 against 27.0, 2048 x 2048 15.5
//     against 18.2
//   m = 2 / 3: 2 x 8192 x 2048 15.1 / 34.8 against 16.7, 2 x 14336 x 4096 70 / 94
//     against 38, Q6_K 2048 x 8192 14.2 / 17.4 against 20, 4096 x 14336 42.8 / 42.1
//     against 35
//   f16 rows as f32: 2 x 8192 x 2048 24.9 / 46.4 against 14.6 / 15.0.  bf16 rows
//     (weights rounded to bf16 in the small-M kernel): 12.2 / 13.9 against 15.1 /
//     15.7, Q6_K 2048 x 8192 29.6 / 33.0 against 18.1 / 18.4, m = 48 36 against 21.
static bool codes_pay(const rq_weight *const *w, int count, int xtype, int64_t m) {
  const int64_t k = w[0]->k;
  int64_t tiles = 0, rows = 0;
  for (int j = 0; j < count; ++j) tiles += ((w[j]->n + 63) / 64) * ((m + 63) / 64), rows += w[j]->n;
  if (m <= 64) {
    if (xtype == RQ_BF16) return m >= 3 && rows * k >= (int64_t)1 << 24 && (m > 32 || k >= 8192);
    return m >= 2 && rows * k >= (m == 2 ? (int64_t)3 << 24 : (int64_t)1 << (m == 3 ? 25 : m <= 16 ? 24 : 23));
  }
  if (xtype == RQ_BF16) return count > 1 ? tiles <= 400 : k >= 4096 && tiles <= 112;
  if (count > 1) return true;
  const bool kfmt = w[0]->qtype == RQ_Q4_K || w[0]->qtype == RQ_Q5_K || w[0]->qtype == RQ_Q6_K;
  return k >= (kfmt ? 896 : 1024);
}

// One weight: the fused kernels, or the generic one for shapes they do not take.
static int linear_one(const rq_weight *w, const void *xa, int xtype, int64_t m, const Out &o, hipStream_t s,
                      WsLease &ws, CodesPack *pack = nullptr) {
  int rc = codes_pay(&w, 1, xtype, m) ? launch_linear_codes(&w, 1, xa, xtype, m, &o, s, ws, pack) : RQ_E_UNSUPPORTED;
  if (rc == RQ_E_UNSUPPORTED) rc = launch_linear_fused(w, xa, xtype, m, o, s, ws);
  if (rc == RQ_E_UNSUPPORTED) rc = launch_linear_generic(w, xa, xtype, m, o, s);
  return rc;
}

int rq_linear_bias(const rq_weight *w, const void *x, int xtype, int64_t m, int64_t k, const void *bias, int btype,
                   void *y, int ytype, void *stream) {
  g_last_error.clear();
  int rc = linear_checks(w, xtype, m, k, bias, btype, ytype);
  if (rc) return rc;
  if (m == 0) return RQ_OK;
  if (!x || !y) return set_error(RQ_E_ARG, "null activation or output");
  rc = hip_check(hipSetDevice(w->device), "hipSetDevice");
  if (rc) return rc;
  const hipStream_t s = as_stream(stream);
  WsLease ws(w->device, s);
  const void *xa = aligned_x(x, xtype, m, k, s, ws, &rc);
  if (!xa) return rc;
  return linear_one(w, xa, xtype, m, Out{y, bias, ytype, btype}, s, ws);
}

int rq_linear(const rq_weight *w, const void *x, int xtype, int64_t m, int64_t k, void *y, int ytype,
              void *stream) {
  return rq_linear_bias(w, x, xtype, m, k, nullptr, RQ_F32, y, ytype, stream);
}

int rq_linear_multi(int count, const rq_weight *const *wts, const void *x, int xtype, int64_t m, int64_t k,
                    const void *const *biases, int btype, void *const *ys, int ytype, void *stream) {
  g_last_error.clear();
  if (count < 0) return set_error(RQ_E_ARG, "negative count %d", count);
  if (count == 0) return RQ_OK;
  if (!wts || !ys) return set_error(RQ_E_ARG, "null weight or output array");
  for (int i = 0; i < count; ++i) {
    const void *b = biases ? biases[i] : nullptr;
    const int rc = linear_checks(wts[i], xtype, m, k, b, btype, ytype);
    if (rc) return rc;
    if (wts[i]->device != wts[0]->device) return set_error(RQ_E_ARG, "weights on different devices");
    if (m > 0 && !ys[i]) return set_error(RQ_E_ARG, "null output %d", i);
  }
  if (m == 0) return RQ_OK;
  if (!x) return set_error(RQ_E_ARG, "null activation");
  int rc = hip_check(hipSetDevice(wts[0]->device), "hipSetDevice");
  if (rc) return rc;
  const hipStream_t s = as_stream(stream);
  WsLease ws(wts[0]->device, s);
  const void *xa = aligned_x(x, xtype, m, k, s, ws, &rc);
  if (!xa) return rc;
  Out outs[kMultiMax];
  // Runs of several formats share one pack of x (q / k in Q4_K, v in Q6_K of
  // 512 rows of 2048: 5 us less).
  CodesPack pack;
  for (int i = 0; i < count; ++i) pack.sums |= wts[i]->qtype == RQ_Q4_K || wts[i]->qtype == RQ_Q5_K;
  for (int i = 0; i < count;) {
    // A run of consecutive weights of one format (at most kMultiMax).
    int j = i + 1;
    while (j < count && j - i < kMultiMax && wts[j]->qtype == wts[i]->qtype) ++j;
    for (int t = i; t < j; ++t) outs[t - i] = Out{ys[t], biases ? biases[t] : nullptr, ytype, btype};
    rc = RQ_E_UNSUPPORTED;
    if (j - i > 1 && codes_pay(wts + i, j - i, xtype, m))
      rc = launch_linear_codes(wts + i, j - i, xa, xtype, m, outs, s, ws, &pack);
    if (j - i > 1 && rc == RQ_E_UNSUPPORTED) rc = launch_linear_multi(wts + i, j - i, xa, xtype, m, outs, s, ws);
    if (rc == RQ_E_UNSUPPORTED) {
      rc = RQ_OK;
      for (int t = i; t < j && !rc; ++t) rc = linear_one(wts[t], xa, xtype, m, outs[t - i], s, ws, &pack);
    }
    if (rc) return rc;
    i = j;
  }
  return RQ_OK;
}

int rq_bias_add(void *y, int ytype, int64_t m, int64_t n, const void *bias, int btype, void *stream) {
  g_last_error.clear();
  if (!valid_ftype(ytype)) return set_error(RQ_E_ARG, "output type %d not supported", ytype);
  if (!valid_ftype(btype)) return set_error(RQ_E_ARG, "bias type %d not supported", btype);
  if (m < 0 || n < 0) return set_error(RQ_E_SHAPE, "bad shape [%lld, %lld]", (long long)m, (long long)n);
  if (m == 0 || n == 0) return RQ_OK;
  if (!y || !bias) return set_error(RQ_E_ARG, "null argument");
  return launch_bias_add(y, ytype, m, n, bias, btype, as_stream(stream));
}

int rq_fp8_quantize(const void *x, int xtype, int64_t m, int64_t k, int mode, uint8_t *xq,
                    float *xscale, void *stream) {
  g_last_error.clear();
  if (!valid_ftype(xtype)) return set_error(RQ_E_ARG, "activation type %d not supported", xtype);
  if (mode != RQ_FP8_UNSCALED && mode != RQ_FP8_PER_TOKEN) return set_error(RQ_E_ARG, "bad fp8 mode %d", mode);
  if (m < 0 || k <= 0) return set_error(RQ_E_SHAPE, "bad shape [%lld, %lld]", (long long)m, (long long)k);
  if (m == 0) return RQ_OK;
  if (!x || !xq || !xscale) return set_error(RQ_E_ARG, "null argument");
  return launch_fp8_quantize(x, xtype, m, k, mode, xq, xscale, as_stream(stream));
}

int rq_fp8_gemm_q(const uint8_t *xq, const float *xscale, int64_t m, const uint8_t *w,
                  const float *w_scale, int64_t n, int64_t k, void *y, int ytype, void *stream) {
  g_last_error.clear();
  if (!valid_ftype(ytype)) return set_error(RQ_E_ARG, "output type %d not supported", ytype);
  if (m < 0 || n <= 0 || k <= 0)
    return set_error(RQ_E_SHAPE, "bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
  if (m == 0) return RQ_OK;
  if (!xq || !w || !y) return set_error(RQ_E_ARG, "null argument");
  return launch_fp8_gemm(xq, xscale, m, w, w_scale, n, k, y, ytype, as_stream(stream));
}

int rq_fp8_gemm(const void *x, int xtype, int64_t m, const uint8_t *w, const float *w_scale,
                int64_t n, int64_t k, void *y, int ytype, int mode, void *stream) {
  g_last_error.clear();
  if (xtype == RQ_F8E4M3)
    return rq_fp8_gemm_q(static_cast<const uint8_t *>(x), nullptr, m, w, w_scale, n, k, y, ytype, stream);
  if (!valid_ftype(xtype)) return set_error(RQ_E_ARG, "activation type %d not supported", xtype);
  if (mode != RQ_FP8_UNSCALED && mode != RQ_FP8_PER_TOKEN) return set_error(RQ_E_ARG, "bad fp8 mode %d", mode);
  if (m < 0 || n <= 0 || k <= 0)
    return set_error(RQ_E_SHAPE, "bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
  if (m == 0) return RQ_OK;
  if (!x || !w || !y) return set_error(RQ_E_ARG, "null argument");
  hipStream_t s = as_stream(stream);
  int dev = 0;
  int rc = hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (rc) return rc;
  const uint64_t qbytes = ((uint64_t)m * (uint64_t)k + 255) & ~(uint64_t)255;
  WsLease ws(dev, s);
  uint8_t *scratch = static_cast<uint8_t *>(ws.get(qbytes + (uint64_t)m * 4, &rc));
  if (!scratch) return rc;
  float *xs = reinterpret_cast<float *>(scratch + qbytes);
  rc = launch_fp8_quantize(x, xtype, m, k, mode, scratch, xs, s);
  if (!rc) rc = launch_fp8_gemm(scratch, xs, m, w, w_scale, n, k, y, ytype, s);
  return rc;
}

int rq_marlin_repack(const void *w, int wtype, const float *scales, int64_t n, int64_t k, uint32_t *packed,
                     void *stream) {
  g_last_error.clear();
  if (!valid_ftype(wtype)) return set_error(RQ_E_ARG, "weight type %d not supported", wtype);
  if (n < 0 || k <= 0) return set_error(RQ_E_SHAPE, "bad shape [%lld, %lld]", (long long)n, (long long)k);
  if (n == 0) return RQ_OK;
  if (!w || !scales || !packed) return set_error(RQ_E_ARG, "null argument");
  return launch_marlin_repack(w, wtype, scales, n, k, packed, as_stream(stream));
}

int rq_marlin_dequant(const uint32_t *packed, const float *scales, int64_t n, int64_t k, float *dev_out,
                      void *stream) {
  g_last_error.clear();
  if (n < 0 || k <= 0) return set_error(RQ_E_SHAPE, "bad shape [%lld, %lld]", (long long)n, (long long)k);
  if (n == 0) return RQ_OK;
  if (!packed || !scales || !dev_out) return set_error(RQ_E_ARG, "null argument");
  return launch_marlin_dequant(packed, scales, n, k, dev_out, as_stream(stream));
}

int rq_marlin_linear(const uint32_t *packed, const float *scales, int64_t n, int64_t k, const void *x, int xtype,
                     int64_t m, void *y, int ytype, void *stream) {
  g_last_error.clear();
  if (!valid_ftype(xtype)) return set_error(RQ_E_ARG, "activation type %d not supported", xtype);
  if (!valid_ftype(ytype)) return set_error(RQ_E_ARG, "output type %d not supported", ytype);
  if (m < 0 || n < 0 || k <= 0)
    return set_error(RQ_E_SHAPE, "bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k);
  if (m == 0 || n == 0) return RQ_OK;
  if (!packed || !scales || !x || !y) return set_error(RQ_E_ARG, "null argument");
  hipStream_t s = as_stream(stream);
  // The codes GEMM (which packs x in a launch of its own) from about 4.2e7
  // multiply-adds: f32, VALU against codes, 8192 x 2048 at m = 2 / 3 / 8 / 32 11.2
  // / 15.1 / 32.5 / 124 against 13.0 / 13.0 / 12.9 / 13.4 us, 2048 x 2048 at m = 8
  // / 16 9.4 / 17.3 against 12.6 / 13.3, 2048 x 1024 at m = 8 / 16 6.3 / 11.1
  // against 9.7 / 9.7, 4096 x 14336 at m = 2 / 3 31.5 / 40.9 against 31.5 / 31.8;
  // 1024 x 512 at m = 32 / 64 9.0 / 16.6 against 10.0 / 13.6.
  if (m > 1 && (double)m * (double)n * (double)k >= 42.0e6) {
    int dev = 0;
    int rc = hip_check(hipGetDevice(&dev), "hipGetDevice");
    if (rc) return rc;
    WsLease ws(dev, s);
    rc = launch_marlin_codes(packed, scales, n, k, x, xtype, m, y, ytype, s, ws);
    if (rc != RQ_E_UNSUPPORTED) return rc;
  }
  return launch_marlin_linear(packed, scales, n, k, x, xtype, m, y, ytype, s);
}

static bool valid_kv_mode(int mode) { return mode == RQ_KV_F16 || mode == RQ_KV_FP8 || mode == RQ_KV_INT8; }

static int kv_quantize(int count, const void *const *t, int ttype, int64_t b, int64_t h, int64_t sd, int mode,
                       void *const *q, float *const *scales, void *stream) {
  g_last_error.clear();
  if (!valid_ftype(ttype)) return set_error(RQ_E_ARG, "input type %d not supported", ttype);
  if (!valid_kv_mode(mode)) return set_error(RQ_E_ARG, "bad kv mode %d", mode);
  if (b < 0 || h < 0 || sd < 0)
    return set_error(RQ_E_SHAPE, "bad shape [%lld, %lld, %lld]", (long long)b, (long long)h, (long long)sd);
  if (h == 0) return RQ_OK;
  for (int i = 0; i < count; ++i)
    if (!scales[i]) return set_error(RQ_E_ARG, "null scales");
  if (b == 0 || sd == 0) {
    // No elements: every head's maximum is 0, so its scale is the floor,
    // written by a kernel (nothing read from host memory at replay time).
    int rc = RQ_OK;
    for (int i = 0; i < count && !rc; ++i)
      rc = launch_kv_fill_scales(scales[i], h, mode == RQ_KV_F16 ? 1.0f : 1e-8f, as_stream(stream));
    return rc;
  }
  for (int i = 0; i < count; ++i)
    if (!t[i] || !q[i]) return set_error(RQ_E_ARG, "null argument");
  int dev = 0;
  const int rc = hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (rc) return rc;
  WsLease ws(dev, as_stream(stream));
  return launch_kv_quantize(count, t, ttype, b, h, sd, mode, q, scales, as_stream(stream), ws);
}

int rq_kv_quantize(const void *t, int ttype, int64_t b, int64_t h, int64_t sd, int mode, void *q, float *scales,
                   void *stream) {
  return kv_quantize(1, &t, ttype, b, h, sd, mode, &q, &scales, stream);
}

int rq_kv_quantize_pair(const void *k, const void *v, int ttype, int64_t b, int64_t h, int64_t sd, int mode, void *kq,
                        void *vq, float *kscales, float *vscales, void *stream) {
  const void *const t[2] = {k, v};
  void *const q[2] = {kq, vq};
  float *const scales[2] = {kscales, vscales};
  return kv_quantize(2, t, ttype, b, h, sd, mode, q, scales, stream);
}

int rq_kv_dequantize(const void *q, int mode, const float *scales, int64_t b, int64_t h, int64_t sd, void *out,
                     int otype, void *stream) {
  g_last_error.clear();
  if (!valid_ftype(otype)) return set_error(RQ_E_ARG, "output type %d not supported", otype);
  if (!valid_kv_mode(mode)) return set_error(RQ_E_ARG, "bad kv mode %d", mode);
  if (b < 0 || h < 0 || sd < 0)
    return set_error(RQ_E_SHAPE, "bad shape [%lld, %lld, %lld]", (long long)b, (long long)h, (long long)sd);
  if (b == 0 || h == 0 || sd == 0) return RQ_OK;
  if (!q || !out || (mode != RQ_KV_F16 && !scales)) return set_error(RQ_E_ARG, "null argument");
  return launch_kv_dequantize(q, mode, scales, b, h, sd, out, otype, as_stream(stream));
}

}  // extern "C"
