// What the library offers the host extension beside it (host_ext.cpp), beyond the C interface.
#pragma once

#include <stdint.h>

// Gated weights of 2^25 .. 2^31 bytes re-laid in their own storage (weight_layout.hip).
extern "C" int phyai_host_relay_gated(void* w, int64_t N, int64_t K, void* scratch, void* stream);
