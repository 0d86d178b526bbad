// Which products pass between the workers of a cooperative tridiagonalisation
// (eigen.hip): m columns, column j with worker j mod nw.
#pragma once

namespace bd {

// Whether y_j is published, and waited for by every worker, at step k. A
// product is needed for j > k. The last nw columns, one of each worker, go on
// being exchanged when they are behind k (their words are read and dropped):
// so every worker publishes something in every step, and a worker that has
// read all of step k + 1 knows that all have read step k, whose slot step
// k + 2 writes again. With the needed products alone a worker whose columns
// are all behind k would publish nothing, the others could run two steps ahead
// of it, and it would wait for a tag that is no longer there.
constexpr bool coop_exchanged(int m, int nw, int k, int j) { return j > k || j >= m - nw; }

}  // namespace bd
