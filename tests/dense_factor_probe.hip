// Test harness: the recovery's factorization of a sequence of matrices as one cell's tries take it (tests/test_dense_factor.py).
// W [count][NS][NS] (row-major, index order) is overwritten with the factors, rows [count][NS] gets their row order,
// exchanged [count] the tries in a row that exchanged rows and cycles [count] the time of each.

extern "C" __global__ void __launch_bounds__(WAVE* REC_WAVES)
    mxc_factor_probe(double* __restrict__ Wg, int* __restrict__ rows, int* __restrict__ exchanged_g,
                     long long* __restrict__ cycles, int count) {
  extern __shared__ double lds[];
  const int lane = (int)(threadIdx.x & (WAVE - 1)), wv = (int)(threadIdx.x / WAVE);
  double* W = lds + L_SIZE;
  double* dinv = W + NS * NS;
  int* pr = (int*)(dinv + 2 * NS);
  volatile int* cmd = pr + NS;
  if (wv != 0) {
    dense_workers(W, pr, dinv, lds + L_DV, cmd, lane, wv);
    return;
  }
  int exchanged = 0;
  for (int b = 0; b < count; b++) {
    for (int e = lane; e < NS * NS; e += WAVE) W[e] = Wg[(size_t)b * NS * NS + e];
    wave_sync();
    const long long start = (long long)__builtin_readcyclecounter();
    dense_factor(W, pr, dinv, lds, cmd, lane, exchanged);
    wave_sync();
    const long long took = (long long)__builtin_readcyclecounter() - start;
    if (lane == 0) {
      exchanged_g[b] = exchanged;
      cycles[b] = took;
    }
    for (int e = lane; e < NS * NS; e += WAVE) Wg[(size_t)b * NS * NS + e] = W[e];
    for (int i = lane; i < NS; i += WAVE) rows[(size_t)b * NS + i] = pr[i];
    wave_sync();
  }
  if (lane == 0) *cmd = DENSE_END;
  __syncthreads();
}
