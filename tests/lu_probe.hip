// Test harness: the LU of one matrix in both layouts (tests/test_lu.py), compiled after a header and common.hip. W: the
// matrix, row-major, elimination order. out: per layout, the factors [NS][NS] as the solves take them (unit L below the
// diagonal, U of the lead rows, U' of the trailing block), then 1 / U_ii [NS]. One workgroup of one wavefront.

extern "C" __global__ void __launch_bounds__(WAVE) mxc_lu_probe(const double* __restrict__ W, const double* __restrict__ b,
                                                                     double* __restrict__ out) {
  extern __shared__ double lds[];
  const int lane = (int)threadIdx.x;
#pragma unroll 1
  for (int which = 0; which < 2; which++) {
    double c[NT], dl, dt;
    LeadRow a21;
    for (int e = lane; e < K0 * NS; e += WAVE) lds[e] = W[e];
    const int row = K0 + (lane < NT ? lane : 0);
#pragma unroll
    for (int k = 0; k < K0; k++) a21[k] = W[row * NS + k];
#pragma unroll
    for (int j = 0; j < NT; j++) c[j] = W[row * NS + K0 + j];
    wave_sync();
    if (which == 0)
      factor_2d(c, a21, dl, dt, lds, lane);
    else
      factor_rows(c, a21, dl, dt, lds, lane);
    wave_sync();
    double* o = out + which * (NS * NS + 4 * NS);
    for (int e = lane; e < K0 * NS; e += WAVE) o[e] = lds[e];
    if (lane < NT) {
#pragma unroll
      for (int k = 0; k < K0; k++) o[row * NS + k] = a21[k];
#pragma unroll
      for (int j = 0; j < NT; j++) o[row * NS + K0 + j] = c[j];
    }
    if (lane < K0) o[NS * NS + lane] = dl;
    if (lane < NT) o[NS * NS + K0 + lane] = dt;
    wave_sync();
    double y1l[1], y1t[1], y2l[2], y2t[2];
    auto get = [&](int v, double& yl, double& yt) {
      yl = lane < K0 ? b[v * NS + lane] : 0.0;
      yt = lane < NT ? b[v * NS + K0 + lane] : 0.0;
    };
    get(0, y1l[0], y1t[0]);
    get(1, y2l[0], y2t[0]);
    get(2, y2l[1], y2t[1]);
    if (which == 0 && BLOCK_SOLVES) {
#pragma unroll
      for (int j = 0; j < NT; j++) c[j] = j == lane ? 0.0 : c[j];
      solve<1, BLOCK_SOLVES>(y1l, y1t, c, a21, dl, dt, lds, lane);
      solve<2, BLOCK_SOLVES>(y2l, y2t, c, a21, dl, dt, lds, lane);
    } else {
      solve<1>(y1l, y1t, c, a21, dl, dt, lds, lane);
      solve<2>(y2l, y2t, c, a21, dl, dt, lds, lane);
    }
    auto put = [&](int v, double yl, double yt) {
      if (lane < K0) o[NS * NS + (1 + v) * NS + lane] = yl;
      if (lane < NT) o[NS * NS + (1 + v) * NS + K0 + lane] = yt;
    };
    put(0, y1l[0], y1t[0]);
    put(1, y2l[0], y2t[0]);
    put(2, y2l[1], y2t[1]);
    wave_sync();
  }
}
