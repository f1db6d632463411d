// Internal interface between the decode entry point and the fast page kernel.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/dartkv.h"

namespace dkv {

struct DecodeParams;

// A page kernel launch that also runs the dense rest (the non-page segments
// and the tail, `chunks` 32-token chunks each), described as the dense
// kernels take it.
struct FusedRest {
  const DecodeParams* rest;
  int chunks;
};

// Loads in flight between a page's value codes and its PV (must be < 16).
int fast_decode_max_loads(int np, int gv);

// LDS bytes one fast-kernel workgroup needs, and one of its waves.
size_t fast_decode_lds_bytes(int np, int gv, int gq);

// Launch the fast kernel over descriptor entries [first, first + count) of
// a.segments (all full 128-token pages with the fast layout), writing splits
// [0, splits) of a workspace whose records hold `split_stride` splits.
int launch_fast_decode(const dkv_decode_args& a, int first, int count, int np, int vg, int splits,
                       int split_stride, hipStream_t stream, const FusedRest* fused = nullptr);

// Uniform pages (KB-bit keys along tokens, VB-bit values along channels):
// the largest load count one wait must cover, and the launch (splits over
// half pages).
int uniform_decode_max_loads(int kb, int vb, int gv);
int launch_uniform_decode(const dkv_decode_args& a, int first, int count, int kb, int vb, int vg, int splits,
                          int split_stride, hipStream_t stream, const FusedRest* fused = nullptr);
// Whether the tile kernel takes a call's page run instead of the page kernels
// (the run is as dkv_decode_args guarantees), and its launch over `count`
// packed entries from `first` on and the n_dense dense entries around them (none
// skipped), writing `splits` records from d.split_offset on.  d.n_total is the
// number of work items: tile_items of those and of the most tokens that a dense
// entry holds.
struct TileLayout {
  int bits, key_group, value_group, promoted;  // promoted 0: uniform pages
};
bool tiles_take_run(const dkv_decode_args& a, int group);
int tile_items(int count, int n_dense, int64_t dense_tokens);
int launch_tile_run(const DecodeParams& d, int first, int count, int n_dense, int splits, const TileLayout& g,
                    hipStream_t stream);

// Whether the tile kernel reads the segments of a decode call outside the page
// kernels' run (checked on the host copies of the descriptors): `count` packed
// ones of one layout from entry `first` of the rest on, the others dense.
struct TileRest {
  int first, count, n_dense, items;
  TileLayout layout;
};
bool tiles_take_rest(const DecodeParams& d, TileRest* rest);
// LDS bytes of one wave of the uniform page kernel.
size_t uniform_decode_wave_lds_bytes(int kb, int vb, int gv);

}  // namespace dkv
