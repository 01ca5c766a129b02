// Internal header of the kernel library: pulls in the public C ABI.
#pragma once
#include "orion_kernels.h"
#include "orion_model_kernels.h"
