// Single-token decode attention at head size 256.
#include "sdpa_decode.h"

namespace kvx {

int launch_decode_256(const decode::DecodeParams& p, int G, int kv, const kvx_h2o_args* hh, hipStream_t st) { return decode::launch_d<256>(p, G, kv, hh, st); }

}  // namespace kvx
