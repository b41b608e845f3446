// The attention of ts_prefill.hip for several chunks, each over keys of its own: the same kernel, which finds its chunk
// first.  Beside the one for a single chunk it is another sixteen instantiations; apart from it both are built,
// and their products' distances checked, side by side.
#define TS_PREFILL_CHUNKS
#include "ts_prefill.hip"
