// The host code of libllminfer_hip.so without a GPU: this program defines the
// HIP runtime calls that the library makes, so device memory is host memory
// (filled with its 16-bit index), copies are copies, and kernel launches are
// recorded by name and not run. Each command prints lines of
// "what name name ..." (tests/test_host_path.py).
#include "llminfer_hip.h"

#include <hip/hip_runtime_api.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>
#include <xmmintrin.h>

namespace {
// (made on first use: the library registers its kernels before main)
std::map<const void *, std::string> &kernels() {
  static std::map<const void *, std::string> m;
  return m;
}
std::vector<std::string> launches;
std::vector<unsigned> grids; // blocks along x of each
size_t largest = SIZE_MAX; // allocations above it fail
hipError_t last = hipSuccess;

// Kernels live in unnamed namespaces: the name follows its length.
std::string base_name(const char *mangled) {
  const char *at = strstr(mangled, "_GLOBAL__N_1");
  if (!at)
    return mangled;
  char *name;
  const long n = strtol(at + 12, &name, 10);
  return std::string(name, n);
}
} // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
  kernels()[host] = base_name(name);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

static thread_local struct {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
} config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  config = {g, b, lds, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
  *g = config.grid, *b = config.block, *lds = config.lds, *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t) {
  launches.push_back(kernels()[f]);
  grids.push_back(grid.x);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  if (n > largest)
    return last = hipErrorOutOfMemory;
  *p = aligned_alloc(256, (n + 255) / 256 * 256);
  for (size_t i = 0; i < n / 2; ++i)
    static_cast<uint16_t *>(*p)[i] = (uint16_t)i;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  memset(d, v, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) {
  *v = 256;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) { // (hipGetDevicePropertiesR0600)
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static unsigned char array[LLMI_HIP_NOALLOC_SCRATCH_BYTES];
  *p = array;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 2;
  return hipSuccess;
}
}

namespace {

void flush_launches(const char *what) {
  printf("%s", what);
  for (const std::string &n : launches)
    printf(" %s", n.c_str());
  printf("\n");
  launches.clear();
  grids.clear();
}

template <typename P> void names(int op, const P &p) {
  printf("names");
  for (unsigned i = 0, n = llmi_hip_dispatch_count(op, &p); i < n; ++i)
    printf(" %s", llmi_hip_kernel_name(op, &p, i));
  printf("\n");
}

// rows rows width: the row norms of a DeltaNet layer, and their blocks.
int rows(char **a) {
  const unsigned n = atoi(a[0]), width = atoi(a[1]);
  void *x = aligned_alloc(256, 256); // (not read)
  auto *u = static_cast<uint16_t *>(x);
  auto *f = static_cast<float *>(x);
  printf("status %d", llmi_hip_l2_norm(u, f, L2Params{n, width, 1e-6f, 1.0f}, nullptr));
  printf(" %d\n", llmi_hip_gated_rms_norm(u, u, f, u, RowParams{n, width, 1e-6f}, nullptr));
  printf("grids");
  for (unsigned g : grids)
    printf(" %u", g);
  printf("\n");
  flush_launches("launches");
  return 0;
}

// conv T channels offset: a 4-tap convolution whose output starts `offset`
// halves past 16-byte alignment.
int conv(char **a) {
  const unsigned T = atoi(a[0]), C = atoi(a[1]);
  auto *u = static_cast<uint16_t *>(aligned_alloc(256, 256)); // (not read)
  printf("status %d\n", llmi_hip_causal_conv(u, u, u, u + atoi(a[2]), ConvParams{T, C, 4, 1},
                                             nullptr));
  flush_launches("launches");
  return 0;
}

// gated T past q_heads kv_heads head_dim rotary place: where the projected
// keys or values lie ("apart", or in an output of the call).
int gated(char **a) {
  const GqaParams p{(unsigned)atoi(a[0]), (unsigned)atoi(a[2]), (unsigned)atoi(a[3]),
                    (unsigned)atoi(a[4]), (unsigned)atoi(a[1])};
  const std::string place = a[6];
  const size_t q = (size_t)p.tokens * p.queryHeads * p.headDim,
               row = (size_t)p.kvHeads * p.headDim, past = p.past * row, kv = p.tokens * row;
  void *qp, *kp, *vp, *kc, *vc, *out, *ws, *w;
  const size_t bytes = llmi_hip_gqa_workspace_bytes(p);
  for (auto [to, n] : {std::pair{&qp, 4 * q}, {&kp, 2 * kv + 16}, {&vp, 2 * kv + 16},
                       {&kc, 2 * (past + kv)}, {&vc, 2 * (past + kv)}, {&out, 2 * q},
                       {&ws, bytes}, {&w, size_t{4} * p.headDim}})
    if (hipMalloc(to, n) != hipSuccess)
      return 1;
  auto u16 = [](void *x) { return static_cast<uint16_t *>(x); };
  uint16_t *k = u16(kp), *v = u16(vp);
  if (place == "keys_in_values")
    k = u16(vc) + past;
  else if (place == "values_in_keys")
    v = u16(kc) + past;
  else if (place == "keys_in_output")
    k = u16(out);
  else if (place == "keys_unaligned")
    k += 1;
  launches.clear();
  const int rc = llmi_hip_gated_attention(u16(qp), k, v, (float *)w, (float *)w, u16(kc), u16(vc),
                                          u16(out), p, atoi(a[5]), 1e-6f, 1e7f, ws, bytes, nullptr);
  printf("status %d\n", rc);
  flush_launches("launches");
  names(LLMI_HIP_OP_GATED_ATTENTION, p);
  return 0;
}

// A two-layer model whose kernels do not run: its logits are what the device
// buffer held, the 65,536 fp16 values.
struct Model {
  std::vector<uint8_t> kinds{0, 1}; // DeltaNet, GQA
  llmi_qwen35_config c{};
  std::vector<llmi_named_weight> weights;
  llmi_qwen35_graph *graph = nullptr;
  llmi_hip_model *session = nullptr;

  explicit Model(uint64_t capacity) {
    c.hidden = 512, c.intermediate = 1024, c.vocabulary = 65536, c.max_positions = 1 << 16;
    c.head_dim = 256, c.q_heads = 4, c.kv_heads = 2, c.rotary_width = 64;
    c.key_heads = 2, c.value_heads = 4, c.key_dim = 128, c.value_dim = 128, c.conv_kernel = 4;
    c.epsilon = 1e-6, c.theta = 1e7, c.w8 = 1;
    c.layer_count = (uint32_t)kinds.size(), c.layer_kinds = kinds.data();
    static unsigned char data[16];
    if (llmi_qwen35_build(&c, 1, 0, capacity, LLMI_LOGITS_ALL, &graph) != LLMI_HIP_OK)
      abort();
    for (size_t i = 0; i < llmi_qwen35_graph_tensor_count(graph); ++i)
      weights.push_back({llmi_qwen35_graph_tensor(graph, i), data, (const uint16_t *)data});
    if (llmi_hip_model_open(&c, weights.data(), weights.size(), capacity, nullptr, &session)) {
      fprintf(stderr, "%s\n", llmi_hip_last_error());
      abort();
    }
  }
  ~Model() {
    llmi_hip_model_close(session);
    llmi_qwen35_graph_destroy(graph);
  }
};

// gqa T past q_heads kv_heads head_dim fused: a CausalGqa, with its KvAppend
// if fused.
int gqa(char **a) {
  const GqaParams p{(unsigned)atoi(a[0]), (unsigned)atoi(a[2]), (unsigned)atoi(a[3]),
                    (unsigned)atoi(a[4]), (unsigned)atoi(a[1])};
  const size_t q = (size_t)p.tokens * p.queryHeads * p.headDim,
               rows = (size_t)(p.past + p.tokens) * p.kvHeads * p.headDim,
               bytes = llmi_hip_gqa_workspace_bytes(p);
  void *m[7];
  const size_t n[7] = {2 * q, 2 * q, 2 * rows, 2 * rows, 2 * rows, 2 * rows, bytes};
  for (int i = 0; i < 7; ++i)
    if (hipMalloc(&m[i], n[i]) != hipSuccess)
      return 1;
  auto u16 = [&](int i) { return static_cast<uint16_t *>(m[i]); };
  const bool fused = atoi(a[5]);
  launches.clear();
  printf("status %d\n",
         fused ? llmi_hip_kv_append_causal_gqa(u16(0), u16(2), u16(3), u16(4), u16(5), u16(1), p,
                                               m[6], bytes, nullptr)
               : llmi_hip_causal_gqa(u16(0), u16(4), u16(5), u16(1), p, m[6], bytes, nullptr));
  flush_launches("launches");
  names(fused ? LLMI_HIP_OP_KV_APPEND_CAUSAL_GQA : LLMI_HIP_OP_CAUSAL_GQA, p);
  return 0;
}

// session past tokens limit: a step of the layer-pair session whose new
// allocations may take up to `limit` bytes each.
int session(char **a) {
  const unsigned past = atoi(a[0]), tokens = atoi(a[1]);
  const llmi_hip_session_config c{past + tokens, 16, 4, 256, 16, 128, 32, 128};
  llmi_hip_session *s = nullptr;
  if (llmi_hip_session_open(&c, nullptr, &s) || llmi_hip_session_restore(s, past))
    return 1;
  void *x; // (read by nothing: the kernels do not run)
  if (hipMalloc(&x, 1 << 20) != hipSuccess)
    return 1;
  auto *f = static_cast<float *>(x);
  auto *u = static_cast<uint16_t *>(x);
  llmi_hip_dispatch records[16];
  size_t count = 0;
  largest = strtoull(a[2], nullptr, 0);
  launches.clear();
  printf("status %d\n", llmi_hip_session_step(s, tokens, f, f, u, f, f, u, u, u, u, u, records, 16,
                                               &count));
  flush_launches("launches");
  printf("names");
  for (size_t i = 0; i < count; ++i)
    printf(" %s", records[i].kernel);
  printf("\npast %u\n", llmi_hip_session_past(s));
  llmi_hip_session_close(s);
  return 0;
}

// model past tokens limit: a step of a two-layer model after `past` rows (in
// steps of 16) whose new allocations may take up to `limit` bytes each, then a
// plan of the same step through llmi_hip_model_run.
int model(char **a) {
  const uint64_t past = atoi(a[0]), tokens = atoi(a[1]);
  Model m(past + 2 * tokens);
  const std::vector<uint32_t> ids(tokens < 16 ? 16 : tokens, 1);
  for (uint64_t p = 0; p < past; p += 16)
    if (llmi_hip_model_step(m.session, ids.data(), 16, LLMI_LOGITS_NONE, nullptr, 0, nullptr))
      return 1;
  llmi_hip_model_step_result r{};
  largest = strtoull(a[2], nullptr, 0);
  launches.clear();
  printf("status %d\n", llmi_hip_model_step(m.session, ids.data(), tokens, LLMI_LOGITS_NONE,
                                            nullptr, 0, &r));
  flush_launches("launches");
  std::vector<llmi_hip_dispatch> records(llmi_hip_model_dispatches(m.session, nullptr, 0));
  llmi_hip_model_dispatches(m.session, records.data(), records.size());
  printf("names");
  for (const auto &d : records)
    printf(" %s", d.kernel);
  printf("\nscratch %llu\ncount %zu\n", (unsigned long long)r.scratch_bytes, r.dispatch_count);
  llmi_hip_plan *plan = nullptr;
  if (llmi_hip_model_plan(m.session, tokens, past + tokens, LLMI_LOGITS_NONE, &plan))
    return 1;
  printf("run %d\n", llmi_hip_model_run(m.session, plan, ids.data(), nullptr));
  flush_launches("again");
  llmi_hip_plan_destroy(plan);
  return 0;
}

double half_value(unsigned h) {
  const int e = h >> 10 & 0x1F, f = h & 0x3FF;
  const double m = e == 0x1F ? (f ? NAN : INFINITY)
                   : e       ? ldexp(1024 + f, e - 25)
                             : ldexp(f, -24);
  return h & 0x8000 ? -m : m;
}

// logits MXCSR: the wrong ones of a step's logits, with the thread's
// floating-point control bits set.
int logits(char **a) {
  Model m(8);
  std::vector<float> out(65536);
  const uint32_t token = 1;
  _mm_setcsr(_mm_getcsr() | (unsigned)strtoul(a[0], nullptr, 0));
  printf("status %d\n", llmi_hip_model_step(m.session, &token, 1, LLMI_LOGITS_LAST, out.data(),
                                            out.size(), nullptr));
  size_t wrong = 0;
  for (unsigned h = 0; h < 65536; ++h) {
    const double want = half_value(h);
    const float exact = (float)want; // (no fp16 value is an fp32 subnormal)
    uint32_t bits, expected;
    memcpy(&bits, &out[h], 4);
    memcpy(&expected, &exact, 4);
    if (std::isnan(want))
      expected = (h & 0x8000u) << 16 | 0x7F800000u | (h & 0x3FFu) << 13;
    wrong += bits != expected;
  }
  printf("wrong %zu\n", wrong);
  return 0;
}

} // namespace

int main(int argc, char **argv) {
  const std::string command = argc > 1 ? argv[1] : "";
  if (command == "gated" && argc == 9)
    return gated(argv + 2);
  if (command == "conv" && argc == 5)
    return conv(argv + 2);
  if (command == "rows" && argc == 4)
    return rows(argv + 2);
  if (command == "gqa" && argc == 8)
    return gqa(argv + 2);
  if (command == "session" && argc == 5)
    return session(argv + 2);
  if (command == "model" && argc == 5)
    return model(argv + 2);
  if (command == "logits" && argc == 3)
    return logits(argv + 2);
  return 2;
}
