// The library's size rules (gcnasm_amd/csrc/routes.hpp) behind C functions, for the tests.
#include "../../gcnasm_amd/csrc/routes.hpp"

extern "C" {
int route_mx_padding_in_launch(long long rows, long long k) { return a8w8::mx_padding_in_launch(rows, k); }
}
