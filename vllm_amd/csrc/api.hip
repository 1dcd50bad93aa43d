// Library-wide pieces of the C ABI: error text, ABI version, cached device facts.
#include "vaq_common.h"

#include <mutex>

namespace vaq {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

static thread_local const VaqTuning* g_tuning = nullptr;
static const VaqTuning g_no_tuning = {};

const VaqTuning& tuning() { return g_tuning ? *g_tuning : g_no_tuning; }
bool tuning_active() { return g_tuning != nullptr; }
// Compute units of the device that the entry point under way on this thread runs on, asked for once a call (0: not yet, or outside of one): the
// rules and plans that a call passes each asked the runtime for the device before.  An eager call of a 2048 x 2048 layer at one row is bound by the host: 6.19 ->
// 6.01 us, with the reservation of LDS that small launches do not need left out (reserve_dynamic_lds).
static thread_local int g_depth = 0, g_call_cus = 0;
TuningScope::TuningScope(const VaqTuning* t) : prev_(g_tuning) {
  g_tuning = t;
  ++g_depth;
}
TuningScope::~TuningScope() {
  g_tuning = prev_;
  if (--g_depth == 0) g_call_cus = 0;
}

// Immutable per-device cache (the only host-visible state of the library).
static int g_cus[64];
static std::once_flag g_cus_once[64];

static int cus_of(int dev) {
  if (dev < 0 || dev >= 64) return -1;
  std::call_once(g_cus_once[dev], [dev] {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) v = -1;
    g_cus[dev] = v;
  });
  return g_cus[dev];
}

int num_cus_current_device() {
  if (g_call_cus > 0) return g_call_cus;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  int c = cus_of(dev);
  c = c > 0 ? c : 256;
  if (g_depth > 0) g_call_cus = c;
  return c;
}

}  // namespace vaq

extern "C" const char* vaq_last_error(void) { return vaq::g_err; }

extern "C" int vaq_abi_version(void) { return 1; }

extern "C" int vaq_num_cus(int device) {
  int c = vaq::cus_of(device);
  if (c <= 0) {
    vaq::set_error("vaq_num_cus: cannot query device %d", device);
    return VAQ_ERR_INVALID_ARG;
  }
  return c;
}
