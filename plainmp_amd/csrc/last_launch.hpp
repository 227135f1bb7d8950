// The launch that ends a call.  A call's completion is remembered by an event
// (calls on different streams wait for one another); recorded on its own, the
// event is a packet of its own behind the kernel, about 3 us a call.  The
// launchers therefore give it to the kernel that ends the call as its stop
// event where the entry point asked for that (call_end, launch.h).  (1,024
// configurations' validity 11.5 -> 8.6 us, 256 rows of evaluate 13.1 -> 10.3.)
#pragma once

#include <hip/hip_ext.h>

#include <tuple>
#include <utility>

#include "launch.h"

namespace pmp {

template <class... P, size_t... I>
inline hipError_t launch_with_stop(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st,
                                   hipEvent_t stop, std::tuple<P...>& args, std::index_sequence<I...>) {
  void* ptrs[] = {(void*)&std::get<I>(args)...};
  return hipExtLaunchKernel((const void*)kernel, grid, block, ptrs, lds, st, nullptr, stop, 0);
}

// The last kernel of a call.  Its own status is returned; a launcher with
// kernels before it asks for theirs first.
template <class... P, class... A>
inline hipError_t launch_last(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t st, A&&... a) {
  if (!call_end.ask) {
    kernel<<<grid, block, lds, st>>>(P(std::forward<A>(a))...);
    return hipGetLastError();
  }
  std::tuple<P...> args{P(std::forward<A>(a))...};
  const hipError_t e =
      launch_with_stop(kernel, grid, block, lds, st, call_end.ask, args, std::index_sequence_for<P...>{});
  if (e == hipSuccess) {
    call_end.done = call_end.ask;
    call_end.ask = nullptr;
  }
  return e;
}

}  // namespace pmp
