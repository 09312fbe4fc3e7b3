// The Cholesky kernels of lk_potrf.hip on the host (hip/hip_runtime.h here).
#include "../../libkriging_amd/csrc/lk_potrf.hip"

using namespace lk;

// Factor the n x n matrix A (n a multiple of 64, column-major) with two block
// columns per launch and plain updates between them; W: the diagonal blocks'
// inverses; cond: their estimates; rb4: 64-row workgroups below the squares.
// order: the waves' order between barriers (8 entries).  Returns the status.
extern "C" int emu_factor(double* A, double* W, double* cond, int n, int mode, const int* order, int lanes_reversed,
                          int rb4) {
  emu::wave_order.assign(order, order + 8);
  emu::lanes_reversed = lanes_reversed != 0;
  const int nblk = n / NB;
  std::vector<double> red(red_size(nblk), 0.0);
  Slot S{};
  S.A = A;
  S.W = W;
  S.red = red.data();
  S.n = S.npad = n;
  S.nblk = nblk;
  SlotParams P{};
  P.active = 1;
  P.mode = mode;
  SlotOut O{};
  Batch B{};
  B.slots = &S;
  B.params = &P;
  B.out = &O;
  B.nslots = 1;
  B.nblk_max = nblk;
  for (int k = 0; k < nblk && O.status == ST_OK; k += 2) {
    const int nb = std::min(2, nblk - k);
    launch_potrf_chain(B, k, nb);
    if (k + nb >= nblk || O.status != ST_OK) break;
    if (rb4)
      emu::launch(k_potrf_rows<4>, dim3(nblk - k - nb, 1), dim3(TPB), B.slots, B.params, B.out, k, nb);
    else
      launch_potrf_rows(B, k, nb);
    if (mode != MODE_FACTOR)
      for (int j = (k + nb) * NB; j < n; ++j)
        for (int q = k * NB; q < (k + nb) * NB; ++q)
          for (int i = j / NB * NB; i < n; ++i) A[i + (size_t)j * n] -= A[i + (size_t)q * n] * A[j + (size_t)q * n];
  }
  for (int k = 0; k < nblk; ++k) cond[k] = red[red_cond_off(nblk) + k];
  return O.status;
}
