// tq_abi.hip -- ABI version and error strings of libtilequant_hip.so.
#include "tq_common.h"

extern "C" int tq_abi_version(void) { return 3; }

extern "C" int64_t tq_stream_capture_id(void* stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(static_cast<hipStream_t>(stream), &status, &id) != hipSuccess) {
    (void)hipGetLastError();   // not a launch's error: the next launch must not report it
    return -1;
  }
  if (status == hipStreamCaptureStatusNone) return 0;
  return status == hipStreamCaptureStatusActive && id != 0 ? (int64_t)id : -1;
}

extern "C" const char* tq_error_string(int code) {
  switch (code) {
    case TQ_OK: return "ok";
    case TQ_ERR_ARG: return "invalid argument (size, stride, null pointer or inconsistent shape)";
    case TQ_ERR_DTYPE: return "unsupported dtype or tile layout code";
    case TQ_ERR_ALIGN: return "tile pointer is not 16-byte aligned";
    case TQ_ERR_WORKSPACE: return "workspace missing or too small";
    default: break;
  }
  if (code > 0) return hipGetErrorString(static_cast<hipError_t>(code));
  return "unknown tilequant error";
}
