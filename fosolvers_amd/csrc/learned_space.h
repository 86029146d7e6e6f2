// Network shape and row buffers of the learned preconditioner (plain C++, so that it can be checked
// without a GPU).
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "learned_slices.h"

namespace fos {

constexpr int NI = 20, NIP = 32, NH = 128, NO = 30, NOP = 32, NBR = 4, NTR = 12;
// The weight-gradient partials of one slice of rows: the layers' [K][N] products, padded as their
// operands are, then the bias gradients
constexpr int PW3 = 0, PW2 = PW3 + NH * NOP, PW1 = PW2 + 2 * NH * NH, PW0 = PW1 + 2 * NH * NH, PB3 = PW0 + NIP * NH;
constexpr int PB2 = PB3 + NOP, PB1 = PB2 + NH, PB0 = PB1 + NH, NPART = PB0 + NH;

// The buffers with a row per cell.  Each one's own size says what it holds (a failed allocation leaves it
// empty), so a call after a failed one allocates what is missing.
template <template <class> class Buf>
struct LearnedSpace {
  // set-up and apply on the mesh, and the same quantities of a training batch
  Buf<float> O, t, kappa;  // O [.][32] network output, t [.][12] = B^ r^ and the weights, kappa [.] output scale
  Buf<double> red;         // reductions
  // set-up only: hidden layers [.][128].  A batch's rows, which hold the neighbours' means as well, are
  // buffers of their own: training does not move what a recorded set-up writes.
  Buf<uint16_t> H0, H1;
  // training only (rows = batch; X also the mesh for fos_learned_inputs)
  Buf<uint16_t> X, HM0, HM1, H2;  // X [.][32] features, HM0/HM1 [.][256] = (h | mean_nb h), H2 [.][128]
  Buf<float> pre0, pre1, pre2, rh, e, ds, part;
  Buf<uint16_t> dO16, dP, dX;  // dO16 [.][32], dP [.][128], dX [.][256]
  Buf<int> bnbr;               // batch-local neighbours [.][4]

  template <class T>
  static int need(Buf<T> &b, size_t count) {
    return b.p && b.n >= count ? 0 : b.alloc(count);
  }
  int apply(size_t n) { return out(n) || need(H0, n * NH) || need(H1, n * NH) ? -1 : 0; }
  int inputs(size_t n) { return need(X, n * NIP) || need(red, n_red(n)) ? -1 : 0; }
  int train(size_t n) {
    return out(n) || inputs(n) || need(HM0, n * 256) || need(HM1, n * 256) || need(H2, n * NH) || need(pre0, n * NH) ||
           need(pre1, n * NH) || need(pre2, n * NH) || need(rh, n * 8) || need(e, n * 8) || need(ds, n * 8) ||
           need(part, slice_room(n) * NPART) || need(dO16, n * NOP) || need(dP, n * NH) || need(dX, n * 256) ||
           need(bnbr, n * NBR) ? -1 : 0;
  }

 private:
  // the state scale's partials (3 of 256 workgroups) or a batch's loss partials
  static size_t n_red(size_t n) { return std::max<size_t>(1024, (n + 255) / 256 + 8); }
  int out(size_t n) { return need(O, n * NOP) || need(t, n * NTR) || need(kappa, n) || need(red, n_red(n)) ? -1 : 0; }
};

}  // namespace fos
