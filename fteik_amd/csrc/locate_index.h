// locate_index.h -- host side of the locator's table index
// (capi_locate_index.cpp), shared with the locator's entry points.
#pragma once
#include <vector>

namespace fteik_capi {

// Picks and weights beyond this are searched without the index: their sums
// may overflow, and a skipped pick's zero term would turn an infinity into
// a NaN.
constexpr float kPlainLimit = 1.0e15f;

// Locates events evnmbr[0..n-1] (1-based) through the index.  0: done, but
// for the events redo (positions in evnmbr), of which the bounds leave too
// much: search these in full; 1: not a search for the index (small, tables
// or picks not finite, no memory): search all in full; 2: GPU error.
int index_search(int n, const int *evnmbr, int *optIndx, double *t0Opt,
                 double *objOpt, std::vector<int> *redo);
// Brings the origin-time work array up to date (capi_locate.cpp).
bool settle_origin_times();
// Frees the index and its work space.
void index_release();

} // namespace fteik_capi
