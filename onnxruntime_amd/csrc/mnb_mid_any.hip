// The many-row form of the streaming kernel for a K with a ragged last chunk, or cut over workgroups (mnb_mid_rows.hip.h).
#include "mnb_mid_rows.hip.h"

hipError_t mnb_mid_launch_any(const void* params, const void* launch, int bits, bool has_zp, int io, hipStream_t s) {
  return launch_rows<true>(*static_cast<const SkinnyParams*>(params), bits, has_zp, io, *static_cast<const MidRowsLaunch*>(launch), s);
}
