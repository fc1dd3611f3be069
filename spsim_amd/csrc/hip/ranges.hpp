// Index arithmetic shared by kernels and host code. Plain C++: constexpr functions
// are device functions too, and a host test compiles them alone.
#pragma once

namespace spsim {

// Where range k of n nearly equal ones of `count` things begins (k = n: where the
// last one ends). The product passes 32 bits from 2^31 / n things on.
constexpr int range_begin(int count, int k, int n) { return (int)((long long)count * k / n); }

}  // namespace spsim
