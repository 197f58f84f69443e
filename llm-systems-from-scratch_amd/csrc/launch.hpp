// Host-side glue shared by the entry points: error reporting.
#pragma once
#include "../../include/mi355_attn.h"

// Records `msg` as the calling thread's last error and returns `code`.
int set_error(int code, const char* msg);

// Whether a grid of so many workgroups can be launched: its threads are counted in 32 bits.
inline bool grid_fits(long long workgroups, int threads) { return workgroups * threads < 1LL << 32; }

// Compute units of the current device; 0 where the runtime does not say.
int device_compute_units();
