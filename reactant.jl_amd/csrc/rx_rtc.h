// Kernel text -> gfx950 code object.
#pragma once
#include <string>

namespace rx {

// The code object of `source` for `arch`; throws rx::Error with the compiler's log where it does not compile.
std::string rtc_compile(const std::string& source, const std::string& arch);

}  // namespace rx
