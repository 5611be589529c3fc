// The recovery kernel: recomputes the cells the guard listed, one wavefront per cell, from their inputs, with the
// call kernel's rates, rhs, Jacobian, stages and step control, but the dense W = I / (gamma h) - Jn - w 1^T factored
// by LU with threshold partial pivoting (the reference's recover kernel, maxichem/kernels/recover.cuh:3-310).

// Dense LU of W (NS x NS, row-major, LDS) in place, shared by the workgroup's REC_WAVES wavefronts (wv: this one's
// index): row k is exchanged with the row of the largest |entry| of column k (ties to the lower row; a NaN is never
// chosen) only when |W_kk| < PIVTAU times it or is not finite. pr[i]: the original row now in row i; dinv[i] =
// 1 / U_ii. Every wavefront reads column k once (rows k + 1 + l (+ WAVE) in lane l's registers, W_kk in all lanes)
// and finds the pivot itself from it, so all take the same branches and meet at the same barriers: the largest
// entry from a wave reduction of the lanes' own largest, then its lowest row from a second one. The pivot and the
// multipliers come from those registers. Wavefront wv updates the blocks of REC_BLOCK columns b = wv, wv +
// REC_WAVES, ... from column k + 1, so every entry takes the same operations in the same order as with one
// wavefront. Wavefront 0 writes column k's multipliers at the start of column k + 1: no other wavefront reads
// column k again, and the next exchange, which moves them, comes after a barrier.
constexpr int REC_BLOCK = 8;
constexpr int REC_ROWS = (NS + WAVE - 2) / WAVE;  // rows below a pivot per lane

__device__ void dense_lu(double* W, int* pr, double* dinv, int lane, int wv) {
  if (wv == 0)
    for (int i = lane; i < NS; i += WAVE) pr[i] = i;
  __syncthreads();
  double l[REC_ROWS];  // column k's multipliers, rows k + 1 + lane + WAVE p
  for (int k = 0; k < NS; k++) {
    if (wv == 0 && k > 0) {
#pragma unroll
      for (int p = 0; p < REC_ROWS; p++) {
        const int i = k + lane + WAVE * p;  // rows below pivot k - 1
        if (i < NS) W[i * NS + k - 1] = l[p];
      }
    }
    double v[REC_ROWS];
#pragma unroll
    for (int p = 0; p < REC_ROWS; p++) {
      const int i = k + 1 + lane + WAVE * p;
      v[p] = i < NS ? W[i * NS + k] : 0.0;
    }
    const double akk = W[k * NS + k];
    double best = -1.0;
    int bi = NS;
    if (lane == 0 && fabs(akk) > best) {  // row k first: each lane sees its rows in increasing order
      best = fabs(akk);
      bi = k;
    }
#pragma unroll
    for (int p = 0; p < REC_ROWS; p++) {
      const int i = k + 1 + lane + WAVE * p;
      if (i < NS && fabs(v[p]) > best) {
        best = fabs(v[p]);
        bi = i;
      }
    }
    const double top = wave_max(best);
    bi = wave_min(best == top ? bi : NS);
    const bool exchange = bi != NS && bi != k && !(fabs(akk) >= PIVTAU * top);
    double piv = akk;
    if (exchange) {
      __syncthreads();  // every wavefront has read column k
      for (int j = lane + WAVE * wv; j < NS; j += WAVE * REC_WAVES) {
        const double a = W[k * NS + j];
        W[k * NS + j] = W[bi * NS + j];
        W[bi * NS + j] = a;
      }
      if (wv == 0 && lane == 0) {
        const int t = pr[k];
        pr[k] = pr[bi];
        pr[bi] = t;
      }
      __syncthreads();
      // row bi's entry is the pivot now, and row bi holds row k's
      const int ob = bi - k - 1, lb = ob % WAVE, pb = ob / WAVE;
      double vb = v[0];
#pragma unroll
      for (int p = 1; p < REC_ROWS; p++) vb = pb == p ? v[p] : vb;
      piv = readlane(vb, lb);
#pragma unroll
      for (int p = 0; p < REC_ROWS; p++) v[p] = (p == pb && lane == lb) ? akk : v[p];
    }
    const double dk = 1.0 / piv;
    if (wv == 0 && lane == 0) dinv[k] = dk;
#pragma unroll
    for (int p = 0; p < REC_ROWS; p++) {
      const int i = k + 1 + lane + WAVE * p;
      l[p] = i < NS ? v[p] * dk : 0.0;
      if (i < NS) {
        for (int j0 = k + 1 + REC_BLOCK * wv; j0 < NS; j0 += REC_BLOCK * REC_WAVES) {
          if (j0 + REC_BLOCK <= NS) {  // a whole block: its loads go out together
            double u[REC_BLOCK], w[REC_BLOCK];
#pragma unroll
            for (int q = 0; q < REC_BLOCK; q++) {
              u[q] = W[k * NS + j0 + q];
              w[q] = W[i * NS + j0 + q];
            }
#pragma unroll
            for (int q = 0; q < REC_BLOCK; q++) W[i * NS + j0 + q] = fma(-l[p], u[q], w[q]);
          } else {
            for (int j = j0; j < NS; j++) W[i * NS + j] = fma(-l[p], W[k * NS + j], W[i * NS + j]);
          }
        }
      }
    }
    __syncthreads();  // the updates are in before the next column is read
  }
}

// The same factors by one wavefront in registers (common.hip's two-dimensional LU, every slot taken), where no pivot
// exchanges rows; returns false and leaves W as it is where the threshold rule would exchange some. lb: the multipliers'
// exchange. A try's W seldom exchanges (6 % of the tries of 367 recovered NCHO cells): this takes 33k cycles where
// dense_lu takes 162k (its columns go through LDS and four barriers).
__device__ __forceinline__ bool dense_lu_2d(double* W, int* pr, double* dinv, double* lb, int lane) {
  lane = opaque_lane(lane);
  const int s = lane & 15, g = lane >> 4;
  LuBlock A;
  auto row = [&](int m) { return (m < LU_ML ? 16 * m : K0 + 16 * (m - LU_ML)) + s; };
  auto col = [&](int t) { return (t < LU_TL ? 4 * t : K0 + 4 * (t - LU_TL)) + g; };
#pragma unroll
  for (int m = 0; m < LU_M; m++) {
    const int i = row(m);
    const double* p = W + (NT == WAVE || i < NS ? i : NS - 1) * NS;  // rows past the matrix read its last one
#pragma unroll
    for (int t = 0; t < LU_T; t++) {
      const double v = p[col(t)];  // a column past the matrix: the next row's, or a reciprocal's place
      A[m][t] = lu_inside(m, t, lane) ? v : 0.0;
    }
  }
  wave_sync();
  if (lu_steps<true>(Steps<NS>{}, A, lb, lane) != 0ull) return false;
  double dg[LU_M];
  lu_diagonal(A, dg, lane);
  if (g == (s & 3)) {
#pragma unroll
    for (int m = 0; m < LU_M; m++)
      if (m < LU_ML ? row(m) < K0 : row(m) < NS) dinv[row(m)] = 1.0 / dg[m];
  }
  for (int i = lane; i < NS; i += WAVE) pr[i] = i;
  wave_sync();
#pragma unroll
  for (int t = 0; t < LU_T; t++) {
    const int j = col(t);
    const double d = dinv[j < NS ? j : NS - 1];
#pragma unroll
    for (int m = 0; m < LU_M; m++) {
      const int i = row(m);
      if (lu_inside(m, t, lane)) W[i * NS + j] = i > j ? A[m][t] * d : A[m][t];
    }
  }
  wave_sync();
  return true;
}

// A recovery workgroup's factorizations. Its first wavefront steps the cell and asks for them through a word in LDS (cmd);
// the others wait for it at a workgroup barrier.
constexpr int DENSE_END = 0, DENSE_ALL = 1, DENSE_REGISTERS = 2;  // cmd: leave; factor W together; the second alone

// What the other wavefronts do until the workgroup's cells are done. The LU in registers (LU_DENSE) runs here, in the second
// wavefront, while the first waits: no register of a try is held around its block, and the kernel needs no scratch memory.
// (As a function called from each try it cost 1.0 KB of it a lane, 530 MB of the device, and 2 % of a recovery's time.)
__device__ __forceinline__ void dense_workers(double* W, int* pr, double* dinv, double* lb, volatile int* cmd, int lane,
                                              int wv) {
  wv = __builtin_amdgcn_readfirstlane(wv);
  for (;;) {
    __syncthreads();
    const int what = __builtin_amdgcn_readfirstlane(*cmd);
    if (what == DENSE_END) return;
    if constexpr (LU_DENSE) {
      if (what == DENSE_REGISTERS) {
        if (wv == 1) dense_lu_2d(W, pr, dinv, lb, lane);
        __syncthreads();
        continue;
      }
    }
    dense_lu(W, pr, dinv, lane, wv);
  }
}

// W's factors, for the first wavefront. exchanged: the cell's last tries in a row whose W exchanged rows (0 at the cell's
// start). After DENSE_EXCHANGES of them the registers are not tried until one exchanges none: two cells that exchange in
// nearly all of their 40,000 tries take 3.86 s, with the registers tried first each time 4.46 s. Fewer would send a cell
// that exchanges now and then (6 % of the tries of 367 recovered NCHO cells) to dense_lu, whose 162k cycles are five
// times the registers' 33k.
constexpr int DENSE_EXCHANGES = 4;

__device__ __forceinline__ void dense_factor(double* W, int* pr, double* dinv, double* ws, volatile int* cmd, int lane,
                                             int& exchanged) {
  if constexpr (LU_DENSE) {
    if (exchanged < DENSE_EXCHANGES) {
      if (lane == 0) {
        *cmd = DENSE_REGISTERS;
        pr[0] = -1;  // the row order is written where the registers have the factors
      }
      __syncthreads();
      __syncthreads();  // the second wavefront has them, or has left W as it was
      if (__builtin_amdgcn_readfirstlane(pr[0]) == 0) {
        exchanged = 0;
        return;
      }
    }
  }
  if (lane == 0) *cmd = DENSE_ALL;
  __syncthreads();
  dense_lu(W, pr, dinv, lane, 0);
  if constexpr (LU_DENSE) {
    bool moved = false;
    for (int i = lane; i < NS; i += WAVE) moved |= pr[i] != i;
    exchanged = __ballot(moved) ? exchanged + 1 : 0;
  }
}

// y <- W^-1 y with dense_lu's factors; y is the vector in LDS (elimination order). Up to ROW_REGISTERS species, this
// lane's row of the factors (row lane, clamped in bounds) is loaded into registers before the substitutions, so the
// chain from step to step is a readlane and an fma with no LDS wait (beyond that the row would not fit the
// registers, and its entries are read in the steps). Rows WAVE and beyond (a second row per lane) read theirs
// DENSE_BATCH steps at a time. Every update is kept by a select, as the substitutions' order fixes the bits.
constexpr int ROW_REGISTERS = 80;
constexpr bool ROW_IN_REGISTERS = NS <= ROW_REGISTERS;
constexpr int DENSE_BATCH = 16;  // steps whose entries of a lane's second row are read together
// Where a lane's row is not in registers its reads stay in their batch: all of them ahead took registers that the function
// must save, and a kernel with saved registers needs scratch memory.

__device__ void dense_solve(const double* W, const int* pr, const double* dinv, double* y, int lane) {
  double a[2];
#pragma unroll
  for (int p = 0; p < 2; p++) a[p] = lane + WAVE * p < NS ? y[pr[lane + WAVE * p]] : 0.0;
  const int r0 = lane < NS ? lane : NS - 1, r1 = lane + WAVE < NS ? lane + WAVE : NS - 1;  // rows in bounds
  double w0[NS];
  if constexpr (ROW_IN_REGISTERS) {
#pragma unroll
    for (int k = 0; k < NS; k++) w0[k] = W[r0 * NS + k];
  }
  const double d0 = dinv[r0], d1 = dinv[r1];
  // a batch of steps' entries of the second row, read for every lane (in bounds) so that no step waits on a branch
  auto second = [&](double (&w)[DENSE_BATCH], int k0, int step) {
#pragma unroll
    for (int i = 0; i < DENSE_BATCH; i++)
      if (NS > WAVE && k0 + i * step >= 0 && k0 + i * step < NS) w[i] = W[r1 * NS + k0 + i * step];
  };
#pragma unroll
  for (int k0 = 0; k0 < NS - 1; k0 += DENSE_BATCH) {
    double w1[DENSE_BATCH];
    if (!ROW_IN_REGISTERS) __builtin_amdgcn_sched_barrier(0);
    second(w1, k0, 1);
#pragma unroll
    for (int i = 0; i < DENSE_BATCH; i++) {
      const int k = k0 + i;
      if (k >= NS - 1) break;
      const double yk = readlane(k < WAVE ? a[0] : a[1], k & (WAVE - 1));
      const double u0 = fma(-(ROW_IN_REGISTERS ? w0[k] : W[r0 * NS + k]), yk, a[0]);
      if (k < WAVE - 1) a[0] = lane > k ? u0 : a[0];
      if (NS > WAVE) {
        const double u1 = fma(-w1[i], yk, a[1]);
        a[1] = lane + WAVE > k && lane + WAVE < NS ? u1 : a[1];
      }
    }
  }
#pragma unroll
  for (int k1 = NS - 1; k1 > 0; k1 -= DENSE_BATCH) {
    double w1[DENSE_BATCH];
    if (!ROW_IN_REGISTERS) __builtin_amdgcn_sched_barrier(0);
    second(w1, k1, -1);
#pragma unroll
    for (int i = 0; i < DENSE_BATCH; i++) {
      const int k = k1 - i;
      if (k <= 0) break;
      const double zk = readlane(k < WAVE ? a[0] * d0 : a[1] * d1, k & (WAVE - 1));
      const double u0 = fma(-(ROW_IN_REGISTERS ? w0[k] : W[r0 * NS + k]), zk, a[0]);
      a[0] = lane < k ? u0 : a[0];
      if (NS > WAVE && k > WAVE) {
        const double u1 = fma(-w1[i], zk, a[1]);
        a[1] = lane + WAVE < k ? u1 : a[1];
      }
    }
  }
  wave_sync();
  if (lane < NS) y[lane] = a[0] * d0;
  if (lane + WAVE < NS) y[lane + WAVE] = a[1] * d1;
  wave_sync();
}

// A lead / trailing vector pair into the LDS vector y (elimination order) and back.
__device__ __forceinline__ void to_lds(double* y, double vl, double vt, int lane) {
  if (lane < K0) y[lane] = vl;
  if (lane < NT) y[K0 + lane] = vt;
  wave_sync();
}

__device__ __forceinline__ void from_lds(const double* y, double& vl, double& vt, int lane) {
  vl = lane < K0 ? y[lane] : 0.0;
  vt = lane < NT ? y[K0 + lane] : 0.0;
  wave_sync();
}

// A workgroup of REC_WAVES wavefronts per listed cell: wavefront 0 steps the cell; the others wait at a workgroup
// barrier for each of its dense factorizations (dense_workers), so every wavefront passes the same barriers.
extern "C" __global__ void __launch_bounds__(WAVE* REC_WAVES)
    mxc_recover(NetP __restrict__ net, const double* __restrict__ x0, const double* __restrict__ Ta,
                const double* __restrict__ Pa, const double* __restrict__ dta, const double* __restrict__ hin,
                double* __restrict__ xout, double* __restrict__ hio, int* __restrict__ doneo,
                double* __restrict__ noko, int* __restrict__ redo, const int* __restrict__ list,
                int* __restrict__ count, double* __restrict__ tries, const double* __restrict__ Jin, double rtol,
                double atol, int max_steps, double* __restrict__ rscratch) {
  const int nfl = count[COUNT_RECOMPUTED];
  if ((int)blockIdx.x >= nfl) return;
  extern __shared__ double lds[];
  const int lane = (int)(threadIdx.x & (WAVE - 1)), wv = (int)(threadIdx.x / WAVE);
  double* ws = lds;
#if RATES_GLOBAL
  double* rk = rscratch + (size_t)blockIdx.x * (2 * NR);  // this workgroup's slot
#else
  double* rk = ws + L_KF;
#endif
  double* W = lds + L_SIZE;
  double* dinv = W + NS * NS;
  double* yv = dinv + NS;
  int* pr = (int*)(yv + NS);
  volatile int* cmd = pr + NS;
  if (wv != 0) {
    dense_workers(W, pr, dinv, ws + L_DV, cmd, lane, wv);
    return;
  }
  double c[NT];
  LeadRow a21;
  int q = (int)blockIdx.x;
  while (q < nfl) {
    const int cell = list[q];
    const double Tc = Ta[cell], dt = dta[cell], nd = Pa[cell] / (KBOLTZ * Tc);
    const double* xr = x0 + (size_t)cell * NS;
    const double* Jc = NJ ? Jin + (size_t)cell * NJ : nullptr;
    // a listed cell passed the call kernel's screen, so it is not screened again
    cell_rates(ws, rk, Tc, nd, net, Jc, lane);
    const double h0 = isfinite(hin[cell]) ? hin[cell] : dt;
    const double m = fmin(h0, dt);
    int ntry = 0, exchanged = 0;
    for (int pass = 0;; pass++) {
      const gptr<int> perm = opaque(net)->perm;
      double Nl = lane < K0 ? xr[perm[lane]] : 0.0, Nt = lane < NT ? xr[perm[K0 + lane]] : 0.0;
      const double start = pass == 0 ? m : fmin(m, dt * pow(REC_RETRY_SPLIT, (double)pass));
      Step s = {fmax(start, H_MIN), 0.0, 0.0, 0.0, 0.0, false};
      int it = dt > 0.0 ? 0 : max_steps;
      while (it < max_steps && s.t < dt * CALL_END) {
        const double ha = fmin(s.h, dt - s.t), igh = 1.0 / (GAMMA * ha), ih = 1.0 / ha;
        double Fl = 0.0, Ft = 0.0, ul = 0.0, ut = 0.0, u0l = 0.0, u0t = 0.0;
        const double ntot = rhs<true>(Nl, Nt, Fl, Ft, u0l, u0t, net, nd, ws, rk, lane);
        jacobian(c, a21, Nl, Nt, u0l, u0t, ntot, ul, ut, net, ws, lane);
        // W = I / (gamma h) - Jn - w 1^T, dense (recover.cuh:124-130)
        to_lds(yv, ul, ut, lane);
        for (int e = lane; e < K0 * NS; e += WAVE) {
          const int i = e / NS;
          W[e] = (e == i * (NS + 1) ? ws[e] + igh : ws[e]) - yv[i];
        }
        if (lane < NT) {
          double* row = W + (K0 + lane) * NS;
#pragma unroll
          for (int k = 0; k < K0; k++) row[k] = a21[k] - ut;
#pragma unroll
          for (int j = 0; j < NT; j++) row[K0 + j] = (j == lane ? c[j] + igh : c[j]) - ut;
        }
        wave_sync();
        dense_factor(W, pr, dinv, ws, cmd, lane, exchanged);
        double K1l, K1t, K2l, K2t, K3l, K3t, K4l, K4t;
        to_lds(yv, Fl, Ft, lane);
        dense_solve(W, pr, dinv, yv, lane);
        from_lds(yv, K1l, K1t, lane);
        to_lds(yv, fma(RODAS_C21 * ih, K1l, Fl), fma(RODAS_C21 * ih, K1t, Ft), lane);
        dense_solve(W, pr, dinv, yv, lane);
        from_lds(yv, K2l, K2t, lane);
        double Yl = Nl + 2.0 * K1l, Yt = Nt + 2.0 * K1t;
        rhs<false>(Yl, Yt, Fl, Ft, u0l, u0t, net, nd, ws, rk, lane);
        to_lds(yv, fma(ih, K1l - K2l, Fl), fma(ih, K1t - K2t, Ft), lane);
        dense_solve(W, pr, dinv, yv, lane);
        from_lds(yv, K3l, K3t, lane);
        Yl = Nl + 2.0 * K1l + K3l;
        Yt = Nt + 2.0 * K1t + K3t;
        rhs<false>(Yl, Yt, Fl, Ft, u0l, u0t, net, nd, ws, rk, lane);
        to_lds(yv, fma(ih, fma(-RODAS_C43, K3l, K1l - K2l), Fl), fma(ih, fma(-RODAS_C43, K3t, K1t - K2t), Ft), lane);
        dense_solve(W, pr, dinv, yv, lane);
        from_lds(yv, K4l, K4t, lane);
        bool ok = false;
        const double en = try_error(Nl, Nt, K1l, K1t, K3l, K3t, K4l, K4t, Yl, Yt, s.t == 0.0, rtol, atol, lane, ok);
        if (ok) {
          Nl = fmax(Yl, 0.0);
          Nt = fmax(Yt, 0.0);
          s.t += ha;
          s.nok += 1.0;
        }
        const double fac = step_factor(en, ok, s.prej, s.pen, s.pha, ha);
        s.h = ha * fac;
        s.prej = !ok;
        s.pen = en;
        s.pha = ha;
        it++;
        ntry++;
      }
      // the guard's test of the result, which goes to the cell's output row (a later pass overwrites it)
      const int dn = s.t >= dt * CALL_END ? 1 : 0;
      const int code = __builtin_amdgcn_readfirstlane(
          guard_wave(Nl, Nt, xr, xout + (size_t)cell * NS, dn != 0, s.nok, atol, net, lane));
      if (code == GUARD_DRIFT && pass < REC_RETRIES) continue;  // only drifted: again, with a smaller first try
      int nx = 0;
      if (lane == 0) {
        hio[cell] = s.h;
        doneo[cell] = code ? 0 : dn;  // done: finished and passing the guard
        noko[cell] = s.nok;
        redo[cell] = code ? 2 : 1;
        if (tries) tries[cell] += (double)ntry;
        atomicAdd(count + (code ? COUNT_STILL_FAILED : COUNT_RECOVERED), 1);
        nx = (int)gridDim.x + atomicAdd(count + COUNT_RECOVERY_QUEUE, 1);
      }
      q = __builtin_amdgcn_readfirstlane(nx);
      break;
    }
  }
  if (lane == 0) *cmd = DENSE_END;
  __syncthreads();  // the other wavefronts leave
}
