// Single-token decode attention at head size 128.
#include "sdpa_decode.h"

namespace kvx {

int launch_decode_128(const decode::DecodeParams& p, int G, int kv, const kvx_h2o_args* hh, hipStream_t st) { return decode::launch_d<128>(p, G, kv, hh, st); }

}  // namespace kvx
