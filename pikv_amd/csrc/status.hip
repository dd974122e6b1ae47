// Status strings and ABI version of libpikv_hip.so.
#include "common.hpp"

extern "C" const char* pikv_status_string(int status) {
  switch (status) {
    case PIKV_OK: return "ok";
    case PIKV_ERR_NULL: return "a required pointer is NULL";
    case PIKV_ERR_SHAPE: return "a dimension is out of range";
    case PIKV_ERR_UNSUPPORTED: return "request not supported by this build";
    case PIKV_ERR_WORKSPACE: return "workspace too small";
    case PIKV_ERR_LAUNCH: return "HIP launch failed";
  }
  return "unknown status";
}

extern "C" int pikv_abi_version(void) { return PIKV_ABI_VERSION; }  // 1.5: + pikv_linear_tiled, pikv_evict_select_h2o, pikv_expert_combine_factors; 1.4: + pikv_quant_append (and the entry points of prefill.hip and moe.hip), pikv_cache_make_room, pikv_quant_scatter_routed
