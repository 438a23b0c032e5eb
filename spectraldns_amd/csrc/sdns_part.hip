// One group of the single-box launchers (SDNS_PART) in one working precision
// (SDNS_REAL); the Makefile compiles this file once per pair.
#include "sdns_launch_impl.hpp"
SDNS_PART(SDNS_REAL)
