// The chained step kernel for one scalar type (a translation unit each, so that they build in parallel).
#include "kpmx_chain_step.hpp"

namespace kpmx {

int launch_chain_c64(const ChainLaunch& L, hipStream_t s) {
    return with_layout<cf32>(L.cols, [&](auto e, auto ew) { return launch_elem<decltype(e), decltype(ew)::value>(L, s); });
}

}  // namespace kpmx
