// Downloads of particle columns (transfer.hip).
#pragma once

#include "ctx.hpp"

namespace mdd {

// device layout -> caller's layout
enum class ColumnKind : int {
    u32,    // u32
    f64,    // f64
    xyz,    // double4 -> 3 f64
    w,      // double4 -> its fourth value
    xyzw,   // double4 -> 4 f64
    ixyz,   // int4 -> 3 i32
    soa32,  // float, component-major (npad apart) -> 3 f64
    soa64,  // double, component-major -> 3 f64
};

struct Column {
    ColumnKind kind;
    const void* dev;
    void* host;
};

// the first n particles of each column, on the context's stream, finished
// before it returns
void download(Ctx& c, const Column* cols, int ncols, int64_t n);
void release_staging(Ctx& c);

}  // namespace mdd
