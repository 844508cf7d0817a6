// Host-only stand-in, see hip_runtime_api.h in this directory.
#pragma once
#include "hip_runtime_api.h"
#define __host__
#define __device__
#define __forceinline__ inline
