// Test harness: the recovery's LU by one wavefront in registers, on matrix b of W [count][NS][NS] (row-major, index
// order), overwritten with the factors where no row would be exchanged; took[b]: whether it was (tests/test_lu.py).

extern "C" __global__ void __launch_bounds__(WAVE) mxc_dense_2d_probe(double* __restrict__ Wg, double* __restrict__ dinvg,
                                                                      int* __restrict__ took) {
  extern __shared__ double lds[];
  const int lane = (int)threadIdx.x, b = (int)blockIdx.x;
  double* W = lds + L_SIZE;
  double* dinv = W + NS * NS;
  int* pr = (int*)(dinv + 2 * NS);
  for (int e = lane; e < NS * NS; e += WAVE) W[e] = Wg[(size_t)b * NS * NS + e];
  wave_sync();
  const bool done = dense_lu_2d(W, pr, dinv, lds + L_DV, lane);
  wave_sync();
  if (lane == 0) took[b] = done ? 1 : 0;
  for (int e = lane; e < NS * NS; e += WAVE) Wg[(size_t)b * NS * NS + e] = W[e];
  for (int i = lane; i < NS; i += WAVE) dinvg[(size_t)b * NS + i] = dinv[i];
}
