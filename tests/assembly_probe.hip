// Test harness: M0's assembly, factorization and solves as a try takes them (which 0: the slots by lu_assemble and
// lu_factor, and the solves by blocks where the network has them) and by rows (which 1), from the same state and rates
// (tests/test_lu_assembly.py), compiled after a header and common.hip. k: the rate coefficients kf, kr [2 NR]; x: the
// state, elimination order; b: three right-hand sides. out, per form: w [NS], the factors [NS][NS], 1 / U_ii [NS] and the
// three solutions [3][NS]. One workgroup of one wavefront.

template <int W>
__device__ __forceinline__ void assembly_form(NetP net, const double* __restrict__ x, const double* __restrict__ b, double nd,
                                              double igh, double* __restrict__ out, double* lds, int lane) {
  const double Nl = lane < K0 ? x[lane] : 0.0, Nt = lane < NT ? x[K0 + lane] : 0.0;
  double c[NT], dl, dt, Fl = 0.0, Ft = 0.0, u0l = 0.0, u0t = 0.0, ul = 0.0, ut = 0.0;
  LeadRow a21;
  const double ntot = rhs<true>(Nl, Nt, Fl, Ft, u0l, u0t, net, nd, lds, lds + L_KF, lane);
  if constexpr (W == 0) {
    LuBlock A;
    lu_assemble<false>(A, igh, Nl, Nt, u0l, u0t, ntot, ul, ut, net, lds, lane);
    lu_factor<BLOCK_SOLVES>(A, c, a21, dl, dt, lds, lane);
  } else {
    jacobian<false>(c, a21, Nl, Nt, u0l, u0t, ntot, ul, ut, net, lds, lane);
    add_diagonal(c, igh, lds, lane);
    factor_rows(c, a21, dl, dt, lds, lane);
  }
  wave_sync();
  double* o = out + W * (NS * NS + 5 * NS);
  auto put = [&](double* at, double vl, double vt) {
    if (lane < K0) at[lane] = vl;
    if (lane < NT) at[K0 + lane] = vt;
  };
  put(o, ul, ut);
  o += NS;
  for (int e = lane; e < K0 * NS; e += WAVE) o[e] = lds[e];
  if (lane < NT) {
    double* row = o + (K0 + lane) * NS;
#pragma unroll
    for (int j = 0; j < K0; j++) row[j] = a21[j];
#pragma unroll
    for (int j = 0; j < NT; j++) row[K0 + j] = c[j];
  }
  o += NS * NS;
  put(o, dl, dt);
  wave_sync();
  constexpr bool BLOCKS = W == 0 && BLOCK_SOLVES;
  double y1l[1] = {lane < K0 ? b[lane] : 0.0}, y1t[1] = {lane < NT ? b[K0 + lane] : 0.0};
  double y2l[2] = {lane < K0 ? b[NS + lane] : 0.0, lane < K0 ? b[2 * NS + lane] : 0.0};
  double y2t[2] = {lane < NT ? b[NS + K0 + lane] : 0.0, lane < NT ? b[2 * NS + K0 + lane] : 0.0};
  solve<1, BLOCKS>(y1l, y1t, c, a21, dl, dt, lds, lane);
  solve<2, BLOCKS>(y2l, y2t, c, a21, dl, dt, lds, lane);
  put(o + NS, y1l[0], y1t[0]);
  put(o + 2 * NS, y2l[0], y2t[0]);
  put(o + 3 * NS, y2l[1], y2t[1]);
  wave_sync();
}

extern "C" __global__ void __launch_bounds__(WAVE)
    mxc_assembly_probe(NetP __restrict__ net, const double* __restrict__ k, const double* __restrict__ x,
                       const double* __restrict__ b, double nd, double igh, double* __restrict__ out) {
  extern __shared__ double lds[];
  const int lane = (int)threadIdx.x;
  for (int i = lane; i < 2 * NR; i += WAVE) lds[L_KF + i] = k[i];
  wave_sync();
  assembly_form<0>(net, x, b, nd, igh, out, lds, lane);
  assembly_form<1>(net, x, b, nd, igh, out, lds, lane);
}
