// C-ABI error state shared by every entry point, and the per-device kernel attributes.
#include <mutex>
#include <set>
#include <utility>

#include "common.h"

namespace msa {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(MSA_ERR_LAUNCH, std::string(what) + ": " + hipGetErrorString(e));
  return MSA_OK;
}

int allow_dynamic_lds(const void* kernel, int bytes, const char* what) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(MSA_ERR_LAUNCH, std::string(what) + ": hipGetDevice: " + hipGetErrorString(e));
  static std::mutex mu;
  static std::set<std::pair<const void*, int>> done;  // (kernel, device) pairs already raised
  std::lock_guard<std::mutex> lock(mu);
  if (done.count({kernel, dev})) return MSA_OK;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return fail(MSA_ERR_LAUNCH, std::string(what) + ": hipFuncSetAttribute: " + hipGetErrorString(e));
  done.insert({kernel, dev});
  return MSA_OK;
}

}  // namespace msa

extern "C" const char* msa_last_error(void) { return msa::g_last_error.c_str(); }

extern "C" int msa_abi_version(void) { return 22; }
