// hull_table.hpp -- the hulls of the 4096 cell keys (HullBits), computed at
// build time by gen_hull_table.cpp: 32 KB, two words a cell, so that a kernel
// holds a hull in two registers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "geom.hpp"

namespace dpx {

static __device__ const HullBits kHullTable[4096] = {
#include "hull_table.inc"
};

}  // namespace dpx
