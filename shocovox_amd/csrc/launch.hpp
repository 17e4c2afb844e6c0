// Kernel launches that answer for themselves.
#pragma once

#include <hip/hip_runtime.h>

#include <tuple>
#include <type_traits>

namespace svo {

// Launches `kernel` and returns this launch's own status. (hipGetLastError after
// a <<<>>> launch returns whatever error the thread's HIP calls left last, an
// earlier one of the caller's included.)
template <class... P, class... A>
inline hipError_t launch(void (*kernel)(P...), dim3 grid, dim3 block, hipStream_t s,
                         const A&... args) {
  static_assert(sizeof...(P) == sizeof...(A), "one argument per parameter");
  std::tuple<std::remove_cv_t<P>...> values(static_cast<P>(args)...);
  return std::apply(
      [&](auto&... v) {
        void* pointers[] = {&v...};
        return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, pointers, 0, s);
      },
      values);
}

}  // namespace svo
