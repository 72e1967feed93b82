// extern "C" access to the scratch memory that bulk inserts share (declared in
// include/warpcore_c.h).
#include "capi_common.hpp"

#include <warpcore/workspace.hpp>

extern "C" uint64_t wc_workspace_bytes(void) { return warpcore::detail::WorkspacePool::instance().bytes_held(); }
extern "C" uint64_t wc_workspace_trim(void) { return warpcore::detail::WorkspacePool::instance().trim(); }
