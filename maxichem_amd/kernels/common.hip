// Shared device arithmetic of the chemistry step: one 64-lane wavefront steps one cell.
//
// A cell's state vectors are held two values per lane: the lead part (elimination row `lane`, valid for lane < K0)
// and the trailing part (row K0 + lane, valid for lane < NT). The trailing block of M0 = I / (gamma h) - Jn sits in
// registers, lane t owning row K0 + t in c[NT], and the same row's lead columns (A21) in a21[K0]; the lead rows sit
// dense in the cell's LDS region (LEAD [K0][NS]). The network header (generated per network) defines the sizes, the
// LDS layout (L_*), the stream rounds and the method's settings.

typedef unsigned int u32;
typedef unsigned long long u64;

// Rodas3 (Sandu et al. 1997): gamma = 1/2 and the stage couplings C21 = 4, C43 = -8/3.
constexpr double GAMMA = 0.5;
constexpr double RODAS_C21 = 4.0;
constexpr double RODAS_C43 = 8.0 / 3.0;
// The Troe factor's published coefficients (Venot et al. 2012, eq. C.2-C.5).
constexpr double TROE_C0 = 0.4;
constexpr double TROE_C1 = 0.67;
constexpr double TROE_N0 = 0.75;
constexpr double TROE_N1 = 1.27;
constexpr double TROE_D = 0.14;
constexpr int REFUSED_COLD = 1;
constexpr int REFUSED_BAD_INPUT = 2;
constexpr int REFUSED_HOT = 3;
constexpr int BROADCAST_WINDOW = 32;  // v_readlane broadcasts of a pivot row in flight ahead of their updates
constexpr int SCHUR_BATCH = 16;  // a lead row's entries read ahead of their Schur updates
constexpr int SMALL_LEAD = 8;  // at most this many lead rows: their factorization and solves are unrolled
typedef double LeadRow[K0 > 0 ? K0 : 1];  // a trailing row's lead columns, one row per lane in registers

// Orders the LDS accesses of the wavefront's lanes: the wave executes in lockstep and LDS serves one wave's accesses
// in issue order, so only the compiler must not move loads and stores across this point.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The places of a queue of pairs that is passed over twice where there are more pairs than wavefronts; once also where
// two passes' places, and the one each wavefront takes past the end, would not fit an int.
__device__ __forceinline__ int queue_places(int pairs, int waves) {
  return pairs > waves && pairs <= (0x7fffffff - waves) / 2 ? 2 * pairs : pairs;
}

// Lane l's value of v, for a wave-uniform l (v_readlane, no LDS).
__device__ __forceinline__ double readlane(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// The LLVM intrinsic behind v_writelane_b32 (clang has no builtin for it): old with lane `lane` set to src, a
// wave-uniform value.
__device__ int writelane_i32(int src, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

// v with lane l's value replaced by x, a wave-uniform value (v_writelane, both 32-bit halves).
__device__ __forceinline__ double writelane(double v, double x, int l) {
  const long long b = __double_as_longlong(v), xb = __double_as_longlong(x);
  const int lo = writelane_i32((int)(xb & 0xffffffffll), l, (int)(b & 0xffffffffll));
  const int hi = writelane_i32((int)(xb >> 32), l, (int)(b >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// v from another lane by a DPP pattern (both 32-bit halves), all lanes active.
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Reductions over the 64 lanes in a fixed order, every lane ending with the same bits: within each row of 16 lanes
// by DPP (pairs, quads, half-rows, rows: each step adds two values in either order, which rounds alike), then the
// four row results in one wave-uniform sum.
constexpr int DPP_XOR1 = 0xb1, DPP_XOR2 = 0x4e, DPP_HALF_MIRROR = 0x141, DPP_MIRROR = 0x140;

__device__ __forceinline__ double wave_sum(double v) {
  v += dpp<DPP_XOR1>(v);
  v += dpp<DPP_XOR2>(v);
  v += dpp<DPP_HALF_MIRROR>(v);
  v += dpp<DPP_MIRROR>(v);
  return (readlane(v, 0) + readlane(v, 16)) + (readlane(v, 32) + readlane(v, 48));
}

// N sums at once, each as wave_sum (the same bits): every DPP step is taken for all N values before the next, so
// the N reductions overlap instead of waiting out each other's latency.
template <int N>
__device__ __forceinline__ void wave_sums(double (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; i++) v[i] += dpp<DPP_XOR1>(v[i]);
#pragma unroll
  for (int i = 0; i < N; i++) v[i] += dpp<DPP_XOR2>(v[i]);
#pragma unroll
  for (int i = 0; i < N; i++) v[i] += dpp<DPP_HALF_MIRROR>(v[i]);
#pragma unroll
  for (int i = 0; i < N; i++) v[i] += dpp<DPP_MIRROR>(v[i]);
#pragma unroll
  for (int i = 0; i < N; i++) v[i] = (readlane(v[i], 0) + readlane(v[i], 16)) + (readlane(v[i], 32) + readlane(v[i], 48));
}

__device__ __forceinline__ double wave_max(double v) {
  v = fmax(v, dpp<DPP_XOR1>(v));
  v = fmax(v, dpp<DPP_XOR2>(v));
  v = fmax(v, dpp<DPP_HALF_MIRROR>(v));
  v = fmax(v, dpp<DPP_MIRROR>(v));
  return fmax(fmax(readlane(v, 0), readlane(v, 16)), fmax(readlane(v, 32), readlane(v, 48)));
}
__device__ __forceinline__ int wave_min(int v) {
  v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_XOR1, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_XOR2, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_HALF_MIRROR, 0xf, 0xf, false));
  v = min(v, __builtin_amdgcn_update_dpp(0, v, DPP_MIRROR, 0xf, 0xf, false));
  return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
             min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// The lane index as an opaque value, taken inside each step of an unrolled loop so that the step's lane masks are
// computed there and not all ahead of the loop, where they would fill the scalar registers.
__device__ __forceinline__ int opaque_lane(int lane) {
  asm volatile("" : "+v"(lane));
  return lane & (WAVE - 1);  // known to be a lane: a test of it against a whole wavefront's rows folds
}

// The cell's LDS region as an opaque place, for the same reason: its addresses made where they are used.
__device__ __forceinline__ double* opaque_lds(double* ws) {
  int zero = 0;
  asm volatile("" : "+s"(zero));
  return ws + zero;
}

// The lane index as an opaque value that the compiler must take after x is computed: a step's lane mask then
// cannot be computed ahead of the step whose value x it follows.
__device__ __forceinline__ int lane_after(int lane, double x) {
  asm volatile("" : "+v"(lane) : "v"(x));
  return lane & (WAVE - 1);
}

// The table pointer p, made opaque to the compiler where it is used, so that the loads and decodes from the
// per-network tables are not hoisted out of the try loop and held in registers across it.
template <typename P>
__device__ __forceinline__ P opaque(P p) {
  asm volatile("" : "+s"(p));
  return p;
}

// a and b materialised here, in this order with the other volatile statements (an empty asm that reads and writes
// them): it keeps a step's values from being computed early or late, which would stretch their live ranges.
__device__ __forceinline__ void pin(double& a, double& b) { asm volatile("" : "+v"(a), "+v"(b)); }
__device__ __forceinline__ void pin(double& a) { asm volatile("" : "+v"(a)); }
// a's next use waits for b (no instruction; an ordering the compiler keeps)
__device__ __forceinline__ void tie(double& a, double b) { asm volatile("" : "+v"(a) : "v"(b)); }
__device__ __forceinline__ void tie(float& a, float b) { asm volatile("" : "+v"(a) : "v"(b)); }

__device__ __forceinline__ bool wave_all(bool p) { return __ballot(!p) == 0ull; }

// A stream word's term: d times the word's coefficient, exactly as fma(coefficient, d, .) takes it: x2 is an exponent
// step, and the sign (the word's bit 31) is XORed into the double's sign bit (one v_bitop3 with its mask; d may be
// negative, a derivative too: an efficiency below 0 makes its reaction's rates negative). No compares and selects, and
// no wait states for condition masks.
static_assert(T_NEG == 31 && SV_NEG == 31, "the streams' sign bit is the word's sign bit");
template <int DBL>
__device__ __forceinline__ double term(u32 w, double d) {
  d = __builtin_amdgcn_ldexp(d, (int)((w >> DBL) & 1u));
  const long long b = __double_as_longlong(d);
  const u32 h = (u32)((u64)b >> 32) ^ (w & 0x80000000u);
  return __longlong_as_double((long long)((u64)h << 32 | (u32)b));
}

// A table pointer in the global address space. Loads through it are global loads, counted by the vector-memory
// counter alone, which the compiler may issue ahead of LDS accesses and wait for only where their values are used.
// Through a plain (flat) pointer, which may address LDS, each load was ordered with the wave's LDS traffic and waited
// for at once: a round of reaction words cost a memory latency.
template <typename T>
using gptr = const __attribute__((address_space(1))) T*;

// The network's tables in device memory, one pointer for every kernel (a function reads the fields it needs through
// opaque(net), so they are loaded where used rather than held in registers across the call).
struct Net {
  gptr<int> perm;      // [NS] network species of elimination row k
  gptr<double> rc;     // [NR][RCW] rate-law rows
  gptr<int> rf;        // [NR] law flags
  gptr<double> nasa;   // [2][NS][9] NASA-9 ranges, elimination order
  gptr<u64> rxe;       // [NR] six species (elimination order, pad NS) and the reaction's first dv slot
  gptr<u32> svw;       // S v stream [SV_ROUNDS][WAVE]
  gptr<u32> rowp;      // [NS] each row's first S v piece | count << 16
  gptr<u32> diagw;     // -Jn streams: diagonal, lead, trailing chunks
  gptr<u32> leadw;
  gptr<u32> chw;
  gptr<double> atoms;  // [NS][NEL] network order
  gptr<int> rord;      // [NR] the order the rate coefficients are computed in (reactions grouped by law)
};
// The Net struct in the constant address space: its fields come by scalar loads, uniform across the wave.
using NetP = const __attribute__((address_space(4))) Net*;

// ---- rate coefficients (the reference's law, collision_limit, gibbs_rt and rate_pair: common.cuh:135-242) ----

// a0, a1, a2: q[0..2], the first Arrhenius term's, which the caller may have loaded ahead
__device__ __forceinline__ double law(gptr<double> __restrict__ q, int fl, double T, double lT, double iT, double nd,
                                      double a0, double a1, double a2) {
  double k = exp(a0 + a1 * lT - a2 * iT);
  if (fl & FL_SECOND_K0) k += exp(q[3] + q[4] * lT - q[5] * iT);
  if (fl & FL_FALLOFF) {
    const double pr = k * nd / exp(q[6] + q[7] * lT - q[8] * iT);
    k = k > 0.0 ? k / (1.0 + pr) : 0.0;  // k0 = 0: no rate, also at Pr = 0 / 0; Pr = inf: the high-pressure 0
#if HAS_TROE
    if ((fl & FL_TROE) && k > 0.0) {
      const double fc = log10((1.0 - q[9]) * exp(-T / q[10]) + q[9] * exp(-T / q[11]) + exp(-q[12] / T));
      const double x = (fl & FL_VM11) ? log10(pr) : log10(pr) - TROE_C0 - TROE_C1 * fc;
      // Pr = 0: Troe's ratio tends to -1 / d, the VM11 one to -inf (F = 1)
      const double y = (fl & FL_VM11) ? x / (TROE_N0 - TROE_N1 * fc)
                                      : (isfinite(x) ? x / (TROE_N0 - TROE_N1 * fc - TROE_D * x) : -1.0 / TROE_D);
      k *= exp10(fc / (1.0 + y * y));
    }
#endif
  }
#if HAS_EFF
  if (fl & FL_EFF) k *= q[13];
#endif
  return k;
}
__device__ __forceinline__ double law(gptr<double> __restrict__ q, int fl, double T, double lT, double iT, double nd) {
  return law(q, fl, T, lT, iT, nd, q[0], q[1], q[2]);
}

// A direction's bimolecular-equivalent rate: M-folded k times nd^(molecules - 2); one molecule without M: none.
__device__ __forceinline__ double bimolecular(int m, bool three_body, double k, double nd) {
  return m >= 2 ? k * (m == 3 ? nd : 1.0) : (three_body ? k / nd : 0.0);
}

// G / RT of one species from its NASA-9 range a at T.
__device__ __forceinline__ double gibbs_rt(gptr<double> __restrict__ a, double T, double lT, double iT) {
  const double T2 = T * T, T3 = T2 * T, T4 = T3 * T;
  const double h = -a[0] * iT * iT + a[1] * lT * iT + a[2] + a[3] * T / 2 + a[4] * T2 / 3 + a[5] * T3 / 4 +
                   a[6] * T4 / 5 + a[7] * iT;
  const double s = -a[0] * iT * iT / 2 - a[1] * iT + a[2] * lT + a[3] * T + a[4] * T2 / 2 + a[5] * T3 / 3 +
                   a[6] * T4 / 4 + a[8];
  return h - s;
}

__device__ __forceinline__ int species_of(u64 w, int m) { return (int)((w >> (8 * m)) & 0xffull); }

// The rate coefficients of every reaction at the cell's T and nd into rk (kf [NR] then kr [NR]; LDS, or the wave's
// slot of global scratch), kept there for the call.
// G / RT (elimination order) goes to the scratch at L_UNION first.
// lmc: the cell's log rate multipliers [NR] or null; each reaction's two coefficients are scaled by exp(lm) after the
// collision limit, a photolysis branch's kf = J exp(lm) (the reference's tangent kernels' rates, ad_common.cuh:136-168)
__device__ __forceinline__ void cell_rates(double* ws, double* rk, double T, double nd, NetP net,
                                           const double* Jc, int lane, const double* lmc = nullptr) {
  ws = opaque_lds(ws);
  lane = opaque_lane(lane);
  net = opaque(net);
  const gptr<double> rc = net->rc;
  const gptr<int> rf = net->rf;
  const gptr<u64> rxe = net->rxe;
  double* g = ws + L_UNION;
  double* kf = rk;
  double* kr = rk + NR;
  const double lT = log(T), iT = 1.0 / T, lKT = log(KBOLTZ * T / P0BAR);
  const gptr<double> cf = net->nasa + (T < NASA_SPLIT_T ? 0 : NS * 9);
  for (int i = lane; i < NS; i += WAVE) g[i] = gibbs_rt(cf + 9 * i, T, lT, iT);
  if (lane == 0) g[NS] = 0.0;
  wave_sync();
  const gptr<int> rord = net->rord;
  // the rounds' table words are loaded a round ahead (the reaction's index two rounds ahead), so that the chain of
  // dependent loads rord -> rf, rxe, rc is not waited on in each round; a lane past NR reads reaction rord[NR - 1]
  auto at = [](int q) { return q < NR ? q : NR - 1; };
  int rn = rord[at(lane)], rnn = rord[at(lane + WAVE)];
  int fn = rf[rn];
  u64 wn = rxe[rn];
  double an0 = rc[RCW * rn], an1 = rc[RCW * rn + 1], an2 = rc[RCW * rn + 2];
#pragma unroll 1
  for (int q = lane; q < NR; q += WAVE) {
    const int r = rn, fl = fn;  // a round's reactions mostly of one law, so it runs the code of few laws
    const u64 w = wn;
    const double a0 = an0, a1 = an1, a2 = an2;
    rn = rnn;
    rnn = rord[at(q + 2 * WAVE)];
    fn = rf[rn];
    wn = rxe[rn];
    an0 = rc[RCW * rn];
    an1 = rc[RCW * rn + 1];
    an2 = rc[RCW * rn + 2];
    double f = 0.0, b = 0.0;
    if (fl & FL_PHOTO) {
      f = Jc[r - NRT];
    } else {
      const double k = law(rc + RCW * r, fl, T, lT, iT, nd, a0, a1, a2);
      const double dg = g[species_of(w, 3)] + g[species_of(w, 4)] + g[species_of(w, 5)] - g[species_of(w, 0)] -
                        g[species_of(w, 1)] - g[species_of(w, 2)];
      const int mf = (fl >> FL_NF_SHIFT) & 3, mr = (fl >> FL_NR_SHIFT) & 3;
      const bool tb = (fl & FL_THREE_BODY) != 0;
      const double c3 = tb ? nd : 1.0;
      f = k * c3;
      b = (k * exp(dg + (double)(mr - mf) * lKT)) * c3;
      const double qb = fmax(bimolecular(mf, tb, f, nd), bimolecular(mr, tb, b, nd));
      if (qb > KCOLL) {  // the collision limit: both directions scaled, their ratio kept
        const double c = KCOLL / qb;
        f *= c;
        b *= c;
      }
    }
    if (lmc) {
      const double e = exp(lmc[r]);
      f *= e;
      b *= e;
    }
    kf[r] = f;
    kr[r] = b;
  }
  wave_sync();
}

// ---- right-hand side and Jacobian ----

// d added to the double at p in LDS, in the order of the wave's LDS accesses (ds_add_f64, rounded as a vector add).
__device__ __forceinline__ void lds_add(double* p, double d) {
  __hip_atomic_fetch_add((__attribute__((address_space(3))) double*)p, d, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// A term stream (the Jacobian's and S v's): each lane adds the terms of whole entries, in their order, to the entries'
// places in dst, which hold 0 before (padding words add 0 to a place of their lane's). The adds are LDS atomics: an
// entry's terms come from one lane, so they are taken in order, and a word costs no running sum, no select and no
// wait: 9 instructions, where a running sum with its selects took 19 (NCHO, cycles of one wavefront per try: the
// Jacobian 23.0k -> 17.4k, the three right-hand sides 21.4k -> 17.9k). The words go a batch of STREAM_BATCH rounds at a
// time: whole batches in a loop, then the last rounds as a batch of their own (the rounds are known when the kernel is
// built). The last batch's words are loaded before the terms of the batch ahead of it are read, those of a stream of one
// batch by its caller, so that it does not wait for them (NCHO, with the rates ahead in rhs: 256 cold cells
// 17.3 -> 16.6 ms, 65,536 settled 7.5 -> 7.15 ms; the loop's words carried from batch to batch as well: no faster, and
// the module takes 62 s to compile instead of 40).
using StreamWords = u32[STREAM_BATCH];

// The words of a stream's rounds from q0 on, at most a batch of them.
template <int ROUNDS, typename WP>
__device__ __forceinline__ void load_words(WP words, int q0, StreamWords& w, int lane) {
#pragma unroll
  for (int i = 0; i < STREAM_BATCH; i++)
    if (q0 + i < ROUNDS) w[i] = words[(q0 + i) * WAVE + lane];
}
// What a stream's caller loads ahead: the words of a stream of one batch.
template <int ROUNDS, typename WP>
__device__ __forceinline__ void load_ahead(WP words, StreamWords& w, int lane) {
  if constexpr (ROUNDS <= STREAM_BATCH) load_words<ROUNDS>(words, 0, w, lane);
}

// w: what load_ahead loaded. next(w): called when the last batch's words are in use, to load another stream's ahead.
template <unsigned IDX_MASK, int DBL, int DEST, unsigned DEST_MASK, int ROUNDS, typename WP, typename Next>
__device__ __forceinline__ void stream_sum(WP words, StreamWords& w, const double* src, double* dst, int lane, Next next) {
  constexpr int LAST = ROUNDS > 0 ? (ROUNDS - 1) / STREAM_BATCH * STREAM_BATCH : 0;  // the last batch's first round
  auto batch = [&](StreamWords& from, int n, auto load) {  // n <= STREAM_BATCH rounds
    StreamWords cur;
    double d[STREAM_BATCH];
#pragma unroll
    for (int i = 0; i < STREAM_BATCH; i++) cur[i] = i < n ? from[i] : 0;
    load();
#pragma unroll
    for (int i = 0; i < STREAM_BATCH; i++)
      if (i < n) d[i] = src[cur[i] & IDX_MASK];
#pragma unroll
    for (int i = 0; i < STREAM_BATCH; i++) {
      if (i >= n) break;
      lds_add(dst + ((cur[i] >> DEST) & DEST_MASK), term<DBL>(cur[i], d[i]));
    }
  };
#pragma unroll 1
  for (int q0 = 0; q0 < LAST; q0 += STREAM_BATCH) {
    StreamWords v;
#pragma unroll
    for (int i = 0; i < STREAM_BATCH; i++) v[i] = words[(q0 + i) * WAVE + lane];
    batch(v, STREAM_BATCH, [&] {
      if (q0 + STREAM_BATCH >= LAST) load_words<ROUNDS>(words, LAST, w, lane);
    });
  }
  batch(w, ROUNDS - LAST, [&] { next(w); });
}

// One Jacobian stream into the cell's LDS: entries of -Jn at their offsets.
template <int ROUNDS, typename WP, typename Next>
__device__ __forceinline__ void jac_stream(WP words, StreamWords& w, const double* DV, double* ws, int lane, Next next) {
  stream_sum<T_IDX_MASK, T_DBL, T_DEST, T_DEST_MASK, ROUNDS>(words, w, DV, ws, lane, next);
}

// The stream words in the workgroup's LDS (WORDS_LDS: the call kernel copies them there at its start, after its
// cells' regions), in the order S v, the Jacobian's diagonal, lead and chunk streams: read with the LDS's latency
// instead of the caches'.
constexpr int W_SV = 0, W_DIAG = SV_ROUNDS * WAVE, W_LEAD = W_DIAG + DIAG_ROUNDS * WAVE;
constexpr int W_CH = W_LEAD + LEAD_ROUNDS * WAVE;
__device__ __forceinline__ const u32* lds_words(const double* ws) {  // ws: this wavefront's cell region
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
  return (const u32*)(ws + (CPW - wv) * L_SIZE);
}

// F = (n_tot / nd) S v(n) at the state Y (lead / trailing parts), u0 = S v / nd; with JAC also the partial
// derivatives dv/dn of every live reaction into DV. Returns n_tot = sum Y.
template <bool JAC, bool LW = false>
__device__ __forceinline__ double rhs(double Yl, double Yt, double& Fl, double& Ft, double& u0l, double& u0t,
                                      NetP net, double nd, double* ws, const double* rk, int lane) {
  ws = opaque_lds(ws);
  lane = opaque_lane(lane);
  const double ntot = wave_sum((lane < K0 ? Yl : 0.0) + (lane < NT ? Yt : 0.0));
  const double xf = nd / ntot, ixf = ntot / nd;
  double* n = ws + L_NVEC;
  if (lane < K0) n[lane] = Yl * xf;
  if (lane < NT) n[K0 + lane] = Yt * xf;
  if (lane == 0) n[NS] = 1.0;  // the padding species of a shorter side
  wave_sync();
  net = opaque(net);
  const gptr<u64> rxe = net->rxe;
  const gptr<int> rf = net->rf;
  const gptr<u32> svw = net->svw;
  const gptr<u32> rowp = net->rowp;
  const double* kf = rk;
  const double* kr = rk + NR;
  double* V = ws + L_V;
  double* DV = ws + L_DV;
  // every round's reaction word (and law flags) loaded first: the loads are in bounds for every lane (the last round's
  // spare lanes read reaction NR - 1), so none waits on the branch that ends a lane's rounds
  u64 wr[RROUNDS];
  int fr[JAC ? RROUNDS : 1];
  double fq[RROUNDS], bq[RROUNDS];
  StreamWords sw;
  auto svp = [&] {
    if constexpr (LW)
      return lds_words(ws) + W_SV;
    else
      return svw;
  }();
  const u32 rpl = rowp[lane < K0 ? lane : 0], rpt = rowp[K0 + (lane < NT ? lane : 0)];  // each row's S v pieces
#pragma unroll
  for (int q = 0; q < RROUNDS; q++) {
    const int r = q * WAVE + lane < NR ? q * WAVE + lane : NR - 1;
    wr[q] = rxe[r];
    if (JAC) fr[q] = rf[r];
    fq[q] = kf[r];
    bq[q] = kr[r];
  }
  load_ahead<SV_ROUNDS>(svp, sw, lane);
#pragma unroll
  for (int q = 0; q < RROUNDS; q++) {
    const int r = q * WAVE + lane;
    if (r >= NR) break;
    const u64 w = wr[q];
    const double n0 = n[species_of(w, 0)], n1 = n[species_of(w, 1)], n2 = n[species_of(w, 2)];
    const double n3 = n[species_of(w, 3)], n4 = n[species_of(w, 4)], n5 = n[species_of(w, 5)];
    const double f = fq[q], b = bq[q];
    V[r] = f * n0 * n1 * n2 - b * n3 * n4 * n5;
    if (JAC) {
      const int fl = fr[JAC ? q : 0];
      if (!(fl & FL_INERT)) {
        int o = (int)(w >> 48);
        const int mf = (fl >> FL_NF_SHIFT) & 3, mr = (fl >> FL_NR_SHIFT) & 3;
        if (mf >= 1) DV[o] = f * n1 * n2;
        if (mf >= 2) DV[o + 1] = f * n0 * n2;
        if (mf >= 3) DV[o + 2] = f * n0 * n1;
        if (!(fl & FL_PHOTO)) {
          o += mf;
          if (mr >= 1) DV[o] = b * n4 * n5;
          if (mr >= 2) DV[o + 1] = b * n3 * n5;
          if (mr >= 3) DV[o + 2] = b * n3 * n4;
        }
      }
    }
  }
  double* part = ws + L_PART;
#pragma unroll
  for (int i = 0; i < NPART; i += WAVE)
    if (i + lane < NPART) part[i + lane] = 0.0;
  if (lane == 0) V[NR] = 0.0;  // the S v stream's padding term
  wave_sync();
  stream_sum<SV_R_MASK, SV_DBL, SV_PIECE, SV_PIECE_MASK, SV_ROUNDS>(svp, sw, V, part, lane, [](StreamWords&) {});
  wave_sync();
  // each row's pieces in order; the reads go out together (a row of fewer pieces than the most reads within part)
  auto row = [&](u32 rp) {
    const int first = (int)(rp & 0xffffu), count = (int)(rp >> 16);
    double v[PIECE_MAX], s = 0.0;
#pragma unroll
    for (int e = 0; e < PIECE_MAX; e++) v[e] = part[e < count ? first + e : 0];
#pragma unroll
    for (int e = 0; e < PIECE_MAX; e++) s = e < count ? s + v[e] : s;
    return s;
  };
  if (K0 > 0) {
    const double s = row(rpl);
    Fl = lane < K0 ? s * ixf : Fl;
    u0l = lane < K0 ? s / nd : u0l;
  }
  const double s = row(rpt);
  Ft = lane < NT ? s * ixf : Ft;
  u0t = lane < NT ? s / nd : u0t;
  wave_sync();
  return ntot;
}

// ---- -Jn from the dv terms that rhs<true> left in DV ----

template <int... K>
struct Seq {};
template <typename T, T... K>
struct IntSeq : Seq<K...> {};
template <int N>
using Steps = __make_integer_seq<IntSeq, int, N>;

template <bool LW, int CH>
__device__ __forceinline__ auto chunk_words(NetP net, const double* ws) {
  if constexpr (LW)
    return lds_words(ws) + W_CH + CH_OFF[CH] * WAVE;
  else
    return opaque(net)->chw + CH_OFF[CH] * WAVE;
}

// One chunk of CHUNK columns of the trailing rows' -Jn, through the staging area (column-major) into sink.chunk, and
// its part of -Jn N. Chunks 0 .. NLCH - 1 hold the lead columns (K0 > 0 means NT == WAVE: every lane has a trailing
// row), the others the trailing columns. cd: the row's own diagonal entry, which the chunk streams do not hold.
// w: the chunk's first words, then the next chunk's.
template <bool LW, int CH, typename Sink>
__device__ __forceinline__ void jac_chunk(Sink& sink, StreamWords& w, double cd, double Nl, double Nt, double& mt,
                                          const double* xv, NetP net, double* ws, int lane) {
  const double* DV = ws + L_DV;
  double* stage = ws + L_STAGE;
  constexpr int C0 = (CH < NLCH ? CH : CH - NLCH) * CHUNK, NC = CH < NLCH ? K0 : NT;  // its first column, of NC
  if (lane < NT) {
#pragma unroll
    for (int j = 0; j < CHUNK; j++) stage[j * NT + lane] = 0.0;
    if (CH >= NLCH && lane / CHUNK == CH - NLCH) stage[(lane % CHUNK) * NT + lane] = cd;
  }
  wave_sync();
  jac_stream<CH_ROUNDS[CH]>(chunk_words<LW, CH>(net, ws), w, DV, ws, lane, [&](StreamWords& v) {
    if constexpr (CH + 1 < NCH) load_ahead<CH_ROUNDS[CH + 1]>(chunk_words<LW, CH + 1>(net, ws), v, lane);
  });
  wave_sync();
  // N_j for -Jn N as wave-uniform values: with few lead rows from the exchange vector (same-address LDS reads, kept in
  // their chunk: hoisted ahead, they would hold a register pair each), else by v_readlane
  double nj[CHUNK], v[CHUNK];
  if constexpr (K0 <= SMALL_LEAD) {
#pragma unroll
    for (int j = 0; j < CHUNK; j++) nj[j] = xv[(CH < NLCH ? 0 : K0) + (C0 + j < NC ? C0 + j : 0)];
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int j = 0; j < CHUNK; j++) v[j] = C0 + j < NC && lane < NT ? stage[j * NT + lane] : 0.0;
  sink.template chunk<CH>(v, stage, lane);
#pragma unroll
  for (int j = 0; j < CHUNK; j++)
    if (C0 + j < NC) mt = fma(v[j], K0 <= SMALL_LEAD ? nj[j] : readlane(CH < NLCH ? Nl : Nt, C0 + j), mt);
  pin(mt);  // taken here: left to its use after the factorization, the chunk's entries would be held until then
}

template <bool LW, typename Sink, int... CH>
__device__ __forceinline__ void jac_chunks(Seq<CH...>, Sink& sink, StreamWords& w, double cd, double Nl, double Nt, double& mt,
                                           const double* xv, NetP net, double* ws, int lane) {
  (jac_chunk<LW, CH>(sink, w, cd, Nl, Nt, mt, xv, net, ws, lane), ...);
}

// -Jn: the lead rows into LEAD (LDS), the trailing rows to sink, from the dv terms in DV; then u = w = S v / nd -
// Jn N / n_tot, the constant-pressure part of the exact Jacobian (lead / trailing parts).
template <bool LW, typename Sink>
__device__ __forceinline__ void jac_assemble(Sink& sink, double Nl, double Nt, double u0l, double u0t, double ntot,
                                             double& ul, double& ut, NetP net, double* ws, int lane) {
  lane = opaque_lane(lane);
  ws = opaque_lds(ws);
  double* DV = ws + L_DV;
  auto dwords = [&] {
    if constexpr (LW)
      return lds_words(ws) + W_DIAG;
    else
      return opaque(net)->diagw;
  }();
  auto lwords = [&] {
    if constexpr (LW)
      return lds_words(ws) + W_LEAD;
    else
      return opaque(net)->leadw;
  }();
  StreamWords w;
  load_ahead<DIAG_ROUNDS>(dwords, w, lane);
  for (int s = lane; s < L_NVEC; s += WAVE) ws[s] = 0.0;  // LEAD
  if (lane < NT) ws[L_DIAG + lane] = 0.0;                   // a species in no reaction has no diagonal term
  if (lane == 0) DV[NDV] = 0.0;                             // the padding words' term
  // the state N in the exchange vector (n's place: free once the dv terms are in DV)
  double* xv = ws + L_NVEC;
  if (lane < K0) xv[lane] = Nl;
  if (lane < NT) xv[K0 + lane] = Nt;
  wave_sync();
  jac_stream<DIAG_ROUNDS>(dwords, w, DV, ws, lane, [&](StreamWords& v) { load_ahead<LEAD_ROUNDS>(lwords, v, lane); });
  jac_stream<LEAD_ROUNDS>(lwords, w, DV, ws, lane, [&](StreamWords& v) {
    load_ahead<CH_ROUNDS[0]>(chunk_words<LW, 0>(net, ws), v, lane);
  });
  wave_sync();
  // -Jn N in FP64: the lead rows through the exchange vector, then the trailing rows chunk by chunk (their lead
  // columns, then the trailing ones)
  double ml = 0.0, mt = 0.0;
  if constexpr (K0 > 0 && K0 <= SMALL_LEAD) {
    // few lead rows: each row times N as this lane's share (its own N entries), summed over the lanes
    double sum[K0 > 0 ? K0 : 1];
#pragma unroll
    for (int i = 0; i < K0; i++)
      sum[i] = (lane < K0 ? ws[i * NS + lane] * Nl : 0.0) + (lane < NT ? ws[i * NS + K0 + lane] * Nt : 0.0);
    wave_sums(sum);
#pragma unroll
    for (int i = 0; i < K0; i++) ml = lane == i ? sum[i] : ml;
  } else if (K0 > 0) {
#pragma unroll 1
    for (int j0 = 0; j0 < NS; j0 += STREAM_BATCH) {  // the lead rows, a batch of columns at a time
      double a[STREAM_BATCH], nv[STREAM_BATCH];
#pragma unroll
      for (int i = 0; i < STREAM_BATCH; i++) {
        const int j = j0 + i;
        a[i] = lane < K0 && j < NS ? ws[lane * NS + j] : 0.0;
        nv[i] = j < NS ? xv[j] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < STREAM_BATCH; i++) ml = fma(a[i], nv[i], ml);
    }
  }
  const double cd = lane < NT ? ws[L_DIAG + lane] : 0.0;
  jac_chunks<LW>(Steps<NCH>{}, sink, w, cd, Nl, Nt, mt, xv, net, ws, lane);
  ul = u0l + ml / ntot;
  ut = lane < NT ? u0t + mt / ntot : 0.0;
  wave_sync();
}

// The trailing rows by lane: their lead columns into a21, the trailing block into c.
template <typename T>
struct RowSink {
  T (&c)[NT];
  LeadRow& a21;
  template <int CH>
  __device__ __forceinline__ void chunk(const double (&v)[CHUNK], const double*, int) {
#pragma unroll
    for (int j = 0; j < CHUNK; j++) {
      if (CH < NLCH && CH * CHUNK + j < K0) a21[CH * CHUNK + j < K0 ? CH * CHUNK + j : 0] = v[j];
      if (CH >= NLCH && (CH - NLCH) * CHUNK + j < NT) c[(CH - NLCH) * CHUNK + j < NT ? (CH - NLCH) * CHUNK + j : 0] = (T)v[j];
    }
  }
};

// -Jn by rows: LEAD (LDS), the trailing rows' lead columns a21 and the trailing block c (registers).
template <bool LW = false, typename T>
__device__ __forceinline__ void jacobian(T (&c)[NT], LeadRow& a21, double Nl, double Nt, double u0l, double u0t,
                                         double ntot, double& ul, double& ut, NetP net, double* ws, int lane) {
  RowSink<T> sink{c, a21};
  jac_assemble<LW>(sink, Nl, Nt, u0l, u0t, ntot, ul, ut, net, ws, lane);
}

// ---- the unpivoted LU of M0 in the elimination order, and its solves ----

// Adds 1 / (gamma h) to M0's diagonal: the lead rows in LDS, the trailing block in registers.
template <typename T>
__device__ __forceinline__ void add_diagonal(T (&c)[NT], double igh, double* ws, int lane) {
  ws = opaque_lds(ws);
  lane = opaque_lane(lane);
  if (lane < K0) ws[lane * NS + lane] += igh;
#pragma unroll
  for (int j = 0; j < NT; j++) c[j] += j == lane ? (T)igh : (T)0;
  wave_sync();
}

// One lead row's Schur update of the trailing block: c_j -= a U_kj, a = this lane's L entry in column k. The row's
// trailing entries come one per lane from a single LDS read and reach every lane by v_readlane (a same-address LDS
// read per entry would wait out the LDS latency once per pair of columns), at most BROADCAST_WINDOW ahead of their
// updates.
template <typename T>
__device__ __forceinline__ void schur_row(T (&c)[NT], double a, const double* ws, int k, int lane) {
  // the row's trailing entries as wave-uniform values from same-address LDS reads (one instruction per pair of
  // entries, where a v_readlane broadcast takes two per entry), SCHUR_BATCH of them issued ahead of their updates
  const double* u = ws + k * NS + K0;
#pragma unroll
  for (int j0 = 0; j0 < NT; j0 += SCHUR_BATCH) {
    double b[SCHUR_BATCH];
#pragma unroll
    for (int i = 0; i < SCHUR_BATCH; i++) b[i] = j0 + i < NT ? u[j0 + i] : 0.0;
#pragma unroll
    for (int i = 0; i < SCHUR_BATCH; i++)
      if (j0 + i < NT) c[j0 + i] = (T)fma(-a, b[i], (double)c[j0 + i]);
    asm volatile("" ::: "memory");  // the next batch's reads stay after this one: hoisted, they hold registers
  }
}

// The Schur update of the trailing block by the lead rows, one lead row at a time. This lane's multipliers go
// through the staging area (free during the factorization) CHUNK at a time, so that the loop over the rows stays
// rolled: unrolled, the compiler would load every row's broadcast values at once.
template <typename T>
__device__ __forceinline__ void schur(T (&c)[NT], const LeadRow& a21, double* ws, int lane) {
  double* stage = ws + L_STAGE;
#pragma unroll
  for (int k0 = 0; k0 < K0; k0 += CHUNK) {
#pragma unroll
    for (int j = 0; j < CHUNK; j++)
      if (k0 + j < K0) stage[j * NT + lane] = a21[k0 + j];
    wave_sync();
#pragma unroll 1
    for (int k = k0; k < (k0 + CHUNK < K0 ? k0 + CHUNK : K0); k++) schur_row(c, stage[(k - k0) * NT + lane], ws, k, lane);
    wave_sync();
  }
}

// LU of the lead columns (right-looking: the lead rows dense in LDS, this lane's trailing row in a21) and the Schur
// update of the trailing block (in T). dl: 1 / U_ii of lead row lane.
template <typename T>
__device__ __forceinline__ void factor_lead(T (&c)[NT], LeadRow& a21, double& dl, double* ws, int lane) {
  dl = 1.0;
  if constexpr (K0 <= SMALL_LEAD) {
    // few lead rows: the steps unrolled
#pragma unroll
    for (int k = 0; k < K0; k++) {
      const double dk = 1.0 / ws[k * NS + k];
      if (lane == k) dl = dk;
      if (lane > k && lane < K0) ws[lane * NS + k] *= dk;
      a21[k] *= dk;
      wave_sync();
#pragma unroll
      for (int i = k + 1; i < K0; i++) {
        const double l = ws[i * NS + k];
#pragma unroll
        for (int j0 = k + 1; j0 < NS; j0 += WAVE) {
          const int j = j0 + lane;
          if (j < NS) ws[i * NS + j] = fma(-l, ws[k * NS + j], ws[i * NS + j]);
        }
      }
#pragma unroll
      for (int j = k + 1; j < K0; j++) a21[j] = fma(-a21[k], ws[k * NS + j], a21[j]);
      wave_sync();
    }
  } else {
    // the steps unrolled for the registers of a21, the lead rows' updates rolled
#pragma unroll
    for (int k = 0; k < K0; k++) {
      const double dk = 1.0 / ws[k * NS + k];
      if (lane == k) dl = dk;
      if (lane > k && lane < K0) ws[lane * NS + k] *= dk;
      a21[k] *= dk;
      wave_sync();
#pragma unroll 1
      for (int i = k + 1; i < K0; i++) {
        const double l = ws[i * NS + k];
        for (int j = k + 1 + lane; j < NS; j += WAVE) ws[i * NS + j] = fma(-l, ws[k * NS + j], ws[i * NS + j]);
      }
#pragma unroll
      for (int j = k + 1; j < K0; j++) a21[j] = fma(-a21[k], ws[k * NS + j], a21[j]);
      wave_sync();
    }
  }
  schur(c, a21, ws, lane);
}

// The trailing block's LU in registers (FP64). dt: 1 / U_ii of trailing row lane.
__device__ __forceinline__ void factor_trailing(double (&c)[NT], double& dt, double* ws, int lane) {
  // the trailing block: at pivot k every lane takes row k's tail from lane k by v_readlane, as wave-uniform values
  // in scalar registers (no LDS round trip, no wait)
  // 1 / U_kk goes through LDS (the union region is free here): a select per step into a register would have the
  // compiler hold every step's reciprocal to the end
  double* dinv = ws + L_UNION;
#pragma unroll
  for (int k = 0; k < NT; k++) {
    const double dk = 1.0 / readlane(c[k], k);
    if (lane == 0) dinv[k] = dk;
    // column k is scaled by 1 / U_kk off the diagonal: below the pivot it becomes the multiplier L_ik, above it
    // U_ik / U_kk, the unit upper factor the backward solve uses (U = U' diag(U_kk))
    const int ln = lane_after(lane, dk);  // the step's lane masks made here, not hoisted and spilled for every step
    if (ln != k) c[k] *= dk;
    const double l = ln > k ? c[k] : 0.0;
#pragma unroll
    for (int j = k + 1; j < NT; j++) {
      // at most BROADCAST_WINDOW of row k's broadcasts ahead of their updates: hoisted further, they would hold up
      // to 126 scalar registers and spill them to vector lanes
      if (j >= k + 1 + BROADCAST_WINDOW) tie(c[j], c[j - BROADCAST_WINDOW]);
      // U_kj is a structural zero of the filled pattern (exactly 0.0): no broadcast, no update
      if ((TRAIL_FILL[k] >> j) & 1ull) c[j] = fma(-l, readlane(c[j], k), c[j]);
    }
  }
  wave_sync();
  dt = lane < NT ? dinv[lane] : 1.0;
  wave_sync();
}

// ---- the LU of the whole of M0 in registers, 16 rows by 4 columns to a register ----
//
// Lane (g, s) = (lane / 16, lane % 16) holds A[m][t], the entry of row s of row slot m and column g of column slot t:
// slots of the lead rows (LU_ML) and columns (LU_TL) first, then of the trailing ones. A pivot's row then sits in one
// lane of each row of 16 lanes, and the updates take it by one DPP row broadcast for all of a lane's rows; a pivot's
// column sits in the 16 lanes of one g, and its multipliers reach the others through LDS, a write and a read per 16
// rows. Each entry takes its updates pivot by pivot, so the factors have the same bits in every layout. Slots that the
// filled pattern keeps zero (LU_ROWS, LU_COLS, LU_LIVE) are left out.
//
// What bounds it is the issue of one wavefront's instructions. By rows (factor_rows) an update costs an fma and the two
// v_readlane of its broadcast; here a broadcast (v_mov_b64_dpp) serves the 16 rows of up to LU_M slots, and a pivot's
// chain (broadcast, reciprocal, LDS round trip) runs beside the previous pivot's updates. Cycles of one wavefront per
// factorization, the lead rows' LU and Schur update included: NCHO (69 species) 40.3k by rows, 24k here; SNCHO (91,
// 27 lead rows, whose LU by rows goes through LDS) 183k and 41k.
typedef double LuBlock[LU_M][LU_T];

// v of lane K of each row of 16 lanes, in the row's lanes; with ROWS only in those rows of lanes, 0 in the others.
template <int K, int ROWS = 0xf>
__device__ __forceinline__ double row_bcast(double v) {
  return __longlong_as_double(
      __builtin_amdgcn_update_dpp(0ll, __double_as_longlong(v), 0x150 + K, ROWS, 0xf, ROWS == 0xf));
}

// 1 / x without the division's scaling steps, which change nothing while x and 1 / x are normal numbers: the same two
// Newton steps and final correction on v_rcp_f64, and the same fixup of zeros, infinities and NaN.
__device__ __forceinline__ double plain_rcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  r = fma(fma(-x, r, 1.0), r, r);
  return __builtin_amdgcn_div_fixup(fma(fma(-x, r, 1.0), r, r), x, 1.0);
}

// Pivot K's place: its row slot and row, its column slot and column.
template <int K>
struct Pivot {
  static constexpr int R = K < K0 ? K : K - K0;
  static constexpr int M = (K < K0 ? 0 : LU_ML) + R / 16, S = R % 16, T = (K < K0 ? 0 : LU_TL) + R / 4, G = R % 4;
};

// Whether pivot K reaches row slot m below it, and column slot t right of it; in a dense matrix it reaches every one.
template <bool DENSE>
__device__ constexpr bool lu_row(int K, int m) { return DENSE || ((LU_ROWS[K] >> m) & 1u); }
template <bool DENSE>
__device__ constexpr bool lu_col(int K, int t) { return DENSE || ((LU_COLS[K] >> t) & 1u); }

// Pivot K's multipliers -l_i K of this lane's rows (0 up to row K) from its column; lb: their exchange, [4][16 LU_M] in
// LDS (each row of lanes writes its own part, the pivot's is read). The column itself keeps its unscaled entries.
// In a dense matrix, swap gathers the lanes that hold an entry below the pivot which the threshold rule would exchange
// with it: |a_KK| not at least PIVTAU |a_iK|.
template <int K, bool DENSE>
__device__ __forceinline__ void lu_pivot(const LuBlock& A, double (&nl)[LU_M], double* lb, int lane, u64& swap) {
  using P = Pivot<K>;
  const double pivot = readlane(A[P::M][P::T], 16 * P::G + P::S);
  const double dk = plain_rcp(pivot);
  const int s = opaque_lane(lane & 15);  // the step's mask made here
  double* mine = lb + (lane >> 4) * (16 * LU_M) + (lane & 15);
  double top = 0.0;
#pragma unroll
  for (int m = P::M; m < LU_M; m++)
    if (lu_row<DENSE>(K, m)) {
      const double x = A[m][P::T] * dk;
      const bool below = m > P::M || s > P::S;
      mine[16 * m] = below ? x : 0.0;
      if (DENSE) top = fmax(top, below ? fabs(A[m][P::T]) : 0.0);
    }
  if (DENSE) swap |= __ballot(!(fabs(pivot) >= PIVTAU * top)) & (0xffffull << (16 * P::G));
  wave_sync();
#pragma unroll
  for (int m = P::M; m < LU_M; m++)
    if (lu_row<DENSE>(K, m)) nl[m] = -lb[P::G * (16 * LU_M) + 16 * m + (lane & 15)];
  wave_sync();
}

// Pivot K's update of column slot t.
template <int K, bool DENSE>
__device__ __forceinline__ void lu_update(LuBlock& A, const double (&nl)[LU_M], int t) {
  using P = Pivot<K>;
  if (!lu_col<DENSE>(K, t)) return;
  const double u =
      t > P::T ? row_bcast<P::S>(A[P::M][t]) : row_bcast<P::S, (0xf << (P::G + 1)) & 0xf>(A[P::M][t]);
#pragma unroll
  for (int m = P::M; m < LU_M; m++)
    if (lu_row<DENSE>(K, m)) A[m][t] = fma(nl[m], u, A[m][t]);
}

// Pivot K's updates, with pivot K + 1's multipliers (a chain of a broadcast, a reciprocal and an LDS round trip) taken
// as soon as its own column is final, while the other columns are updated.
template <int K, bool DENSE>
__device__ __forceinline__ void lu_step(LuBlock& A, double (&nl)[LU_M], double* lb, int lane, u64& swap) {
  __builtin_amdgcn_sched_barrier(0);
  constexpr int TN = Pivot<K + 1 < NS ? K + 1 : K>::T;
  double next[LU_M];
  if constexpr (K + 1 < NS) {
    lu_update<K, DENSE>(A, nl, TN);
    lu_pivot<K + 1, DENSE>(A, next, lb, lane, swap);
  }
#pragma unroll
  for (int t = Pivot<K>::T; t < LU_T; t++)
    if (t != TN) lu_update<K, DENSE>(A, nl, t);
  if constexpr (K + 1 < NS) {
#pragma unroll
    for (int m = 0; m < LU_M; m++) nl[m] = next[m];
  }
}

// Every pivot in turn; returns swap (0 but in a dense matrix).
template <bool DENSE, int... K>
__device__ __forceinline__ u64 lu_steps(Seq<K...>, LuBlock& A, double* lb, int lane) {
  double nl[LU_M];
  u64 swap = 0;
  lu_pivot<0, DENSE>(A, nl, lb, lane, swap);
  (lu_step<K, DENSE>(A, nl, lb, lane, swap), ...);
  return swap;
}

// The diagonal after the LU, by row slot: row s of a row slot has it in column slot s / 4 of the slot's four, in the
// lanes of g = s % 4 (the other lanes' values are not the diagonal's).
__device__ __forceinline__ void lu_diagonal(const LuBlock& A, double (&dg)[LU_M], int lane) {
  const int q = (lane & 15) >> 2;
#pragma unroll
  for (int m = 0; m < LU_M; m++) {
    const int t0 = m < LU_ML ? 4 * m : LU_TL + 4 * (m - LU_ML), last = m < LU_ML ? LU_TL : LU_T;
    dg[m] = A[m][t0];
#pragma unroll
    for (int u = 1; u < 4; u++)
      if (t0 + u < last) dg[m] = q == u ? A[m][t0 + u] : dg[m];
  }
}

// A lane's place of slot (m, t) in a chunk of columns, column-major with LU_STRIDE doubles a column for the trailing
// rows' slots, or in the lead rows.
struct LuPlace {
  double *chunk, *lead;
  __device__ __forceinline__ LuPlace(double* ws, int lane)
      : chunk(ws + L_DV + (lane >> 4) * LU_STRIDE + (lane & 15)), lead(ws + (lane & 15) * NS + (lane >> 4)) {}
  __device__ __forceinline__ double* at(int m, int t, int t0) const {
    return m < LU_ML ? lead + 16 * m * NS + (t < LU_TL ? 4 * t : K0 + 4 * (t - LU_TL))
                     : chunk + 4 * (t - t0) * LU_STRIDE + 16 * (m - LU_ML);
  }
};

// Whether this lane's entry of slot (m, t) is inside the matrix (the slots' last rows and columns may not be).
__device__ __forceinline__ bool lu_inside(int m, int t, int lane) {
  const int i = m < LU_ML ? 16 * m : 16 * (m - LU_ML), j = t < LU_TL ? 4 * t : 4 * (t - LU_TL);
  const int ni = m < LU_ML ? K0 : NT, nj = t < LU_TL ? K0 : NT;
  return (i + 16 <= ni || i + (lane & 15) < ni) && (j + 4 <= nj || j + (lane >> 4) < nj);
}

// A from the rows by lane (c, a21, and the lead rows in LDS), for a caller that has the matrix by rows, as the LU's tests
// do (a try assembles straight into the slots, lu_assemble): columns pass LU_CHUNK slots at a time through the cell's LDS
// from its dv terms on, which no later part of a try reads.
__device__ __forceinline__ void lu_load(LuBlock& A, const double (&c)[NT], const LeadRow& a21, double* ws, int lane) {
  const LuPlace p(ws, lane);
  double* buf = ws + L_DV;
#pragma unroll
  for (int t0 = 0; t0 < LU_T; t0 += LU_CHUNK) {
    if (lane < NT) {
#pragma unroll
      for (int t = t0; t < t0 + LU_CHUNK && t < LU_T; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const int j = t < LU_TL ? 4 * t + g : 4 * (t - LU_TL) + g;
          if (t < LU_TL ? j < K0 : j < NT)
            buf[(4 * (t - t0) + g) * LU_STRIDE + lane] = t < LU_TL ? a21[j < K0 ? j : 0] : c[j < NT ? j : 0];
        }
    }
    wave_sync();
#pragma unroll
    for (int m = 0; m < LU_M; m++)
#pragma unroll
      for (int t = t0; t < t0 + LU_CHUNK && t < LU_T; t++) {
        A[m][t] = 0.0;
        if ((LU_LIVE[m] >> t) & 1u) {
          const double v = *p.at(m, t, t0);  // outside the matrix: some place of the cell's
          A[m][t] = lu_inside(m, t, lane) ? v : 0.0;
        }
      }
    wave_sync();
  }
}

// The factors out of A: 1 / U_ii of lead row lane (dl) and of trailing row lane (dt); each column times its 1 / U_jj
// below the diagonal (L) and, in the trailing rows, above it (U' = U diag(1 / U_jj)); and the rows back to their lanes.
// ZERO: the trailing diagonal as 0 (for solve_blocks), else U_ii.
template <bool ZERO>
__device__ __forceinline__ void lu_store(LuBlock& A, double (&c)[NT], LeadRow& a21, double& dl, double& dt, double* ws,
                                         int lane) {
  const LuPlace p(ws, lane);
  const int s = lane & 15, g = lane >> 4;
  double* buf = ws + L_DV;
  double dg[LU_M];
  lu_diagonal(A, dg, lane);
  if (g == (s & 3)) {
#pragma unroll
    for (int m = 0; m < LU_M; m++) buf[16 * m + s] = dg[m];
  }
  wave_sync();
  double* dinv = buf + 16 * LU_M;  // by column, a slot's four together
  dl = lane < K0 ? 1.0 / buf[lane < K0 ? lane : 0] : 1.0;
  dt = lane < NT ? 1.0 / buf[16 * LU_ML + lane] : 1.0;
  if (lane < 4 * LU_TL) dinv[lane] = dl;
  dinv[4 * LU_TL + lane] = dt;
  wave_sync();
#pragma unroll
  for (int t = 0; t < LU_T; t++) {
    const double d = dinv[4 * t + g];
#pragma unroll
    for (int m = 0; m < LU_M; m++) {
      const bool lead_u = m < LU_ML && (t >= LU_TL || t / 4 > m);  // a lead row's slot right of its diagonal
      if (!((LU_LIVE[m] >> t) & 1u) || lead_u) continue;
      const bool diag = m < LU_ML ? t < LU_TL && t / 4 == m : t >= LU_TL && (t - LU_TL) / 4 == m - LU_ML;
      const int j = 4 * (m < LU_ML ? t & 3 : (t - LU_TL) & 3) + g;  // the column's row in a diagonal slot
      A[m][t] *= !diag || s > j || (m >= LU_ML && s != j) ? d : 1.0;
      if (ZERO && diag && m >= LU_ML) A[m][t] = s == j ? 0.0 : A[m][t];
    }
  }
  wave_sync();
#pragma unroll
  for (int t0 = 0; t0 < LU_T; t0 += LU_CHUNK) {
#pragma unroll
    for (int m = 0; m < LU_M; m++)
#pragma unroll
      for (int t = t0; t < t0 + LU_CHUNK && t < LU_T; t++)
        if (m >= LU_ML || (((LU_LIVE[m] >> t) & 1u) && lu_inside(m, t, lane))) *p.at(m, t, t0) = A[m][t];
    wave_sync();
    if (lane < NT) {
#pragma unroll
      for (int t = t0; t < t0 + LU_CHUNK && t < LU_T; t++)
#pragma unroll
        for (int h = 0; h < 4; h++) {
          const int j = t < LU_TL ? 4 * t + h : 4 * (t - LU_TL) + h;
          const double v = buf[(4 * (t - t0) + h) * LU_STRIDE + lane];
          if (t < LU_TL) {
            if (j < K0) a21[j < K0 ? j : 0] = v;
          } else if (j < NT) {
            c[j < NT ? j : 0] = v;
          }
        }
    }
    wave_sync();
  }
}

// The trailing rows' slots, from the staging area.
struct LuSink {
  LuBlock& A;
  template <int CH>
  __device__ __forceinline__ void chunk(const double (&)[CHUNK], const double* stage, int lane) {
    constexpr int T0 = CH < NLCH ? CH * (CHUNK / 4) : LU_TL + (CH - NLCH) * (CHUNK / 4), END = CH < NLCH ? LU_TL : LU_T;
    const double* p = stage + (lane >> 4) * NT + (lane & 15);
#pragma unroll
    for (int t = T0; t < T0 + CHUNK / 4 && t < END; t++)
#pragma unroll
      for (int m = LU_ML; m < LU_M; m++) {
        A[m][t] = 0.0;
        if ((LU_LIVE[m] >> t) & 1u) {
          const double v = p[4 * (t - T0) * NT + 16 * (m - LU_ML)];  // outside the matrix: some place of the cell's
          A[m][t] = lu_inside(m, t, lane) ? v : 0.0;
        }
      }
  }
};

// M0 = igh - Jn into A's slots, LEAD, and u as jacobian's.
template <bool LW>
__device__ __forceinline__ void lu_assemble(LuBlock& A, double igh, double Nl, double Nt, double u0l, double u0t,
                                            double ntot, double& ul, double& ut, NetP net, double* ws, int lane) {
  LuSink sink{A};
  jac_assemble<LW>(sink, Nl, Nt, u0l, u0t, ntot, ul, ut, net, ws, lane);
  lane = opaque_lane(lane);
  const LuPlace p(opaque_lds(ws), lane);
  const int s = lane & 15, g = lane >> 4;
#pragma unroll
  for (int m = 0; m < LU_ML; m++)
#pragma unroll
    for (int t = 0; t < LU_T; t++) {
      A[m][t] = 0.0;
      if ((LU_LIVE[m] >> t) & 1u) {
        const double v = *p.at(m, t, 0);
        A[m][t] = lu_inside(m, t, lane) ? v : 0.0;
      }
    }
#pragma unroll
  for (int m = 0; m < LU_M; m++) {
    const int t0 = m < LU_ML ? 4 * m : LU_TL + 4 * (m - LU_ML), last = m < LU_ML ? LU_TL : LU_T;
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (t0 + u < last) A[m][t0 + u] += s == 4 * u + g ? igh : 0.0;
  }
  wave_sync();
}

// The LU of A into the rows by lane, and the reciprocals of its diagonal.
template <bool ZERO>
__device__ __forceinline__ void lu_factor(LuBlock& A, double (&c)[NT], LeadRow& a21, double& dl, double& dt, double* ws,
                                          int lane) {
  lane = opaque_lane(lane);
  ws = opaque_lds(ws);
  lu_steps<false>(Steps<NS>{}, A, ws + L_DV, lane);
  wave_sync();
  lu_store<ZERO>(A, c, a21, dl, dt, opaque_lds(ws), opaque_lane(lane));
}

__device__ __forceinline__ void factor_2d(double (&c)[NT], LeadRow& a21, double& dl, double& dt, double* ws, int lane) {
  LuBlock A;
  lu_load(A, c, a21, opaque_lds(ws), opaque_lane(lane));
  lu_factor<false>(A, c, a21, dl, dt, ws, lane);
}

// The LU of M0 by rows: the lead columns (right-looking, dense in LDS), the Schur update of the trailing block, then
// the trailing block in registers. dl: 1 / U_ii of lead row lane; dt: of trailing row lane.
__device__ __forceinline__ void factor_rows(double (&c)[NT], LeadRow& a21, double& dl, double& dt, double* ws,
                                            int lane) {
  factor_lead(c, a21, dl, ws, lane);
  factor_trailing(c, dt, ws, lane);
}

__device__ __forceinline__ void factor(double (&c)[NT], LeadRow& a21, double& dl, double& dt, double* ws, int lane) {
  if constexpr (LU_2D)
    factor_2d(c, a21, dl, dt, ws, lane);
  else
    factor_rows(c, a21, dl, dt, ws, lane);
}

// y <- M0^-1 y for NV vectors (lead / trailing parts), with factor's factors, in three parts: the lead columns of L,
// the trailing block, the lead rows of U.
constexpr int LEAD_BATCH = 14;  // lead columns read ahead of their steps

template <int NV>
__device__ __forceinline__ void solve_lead_forward(double (&yl)[NV], double (&yt)[NV], const LeadRow& a21,
                                                   const double* ws, int lane) {
  const double* row = ws + (lane < K0 ? lane : 0) * NS;  // in bounds for every lane, so that no read waits on a branch
#pragma unroll
  for (int k0 = 0; k0 < K0; k0 += LEAD_BATCH) {  // unit L, lead columns (the trailing rows' entries in a21)
    double l[LEAD_BATCH];
#pragma unroll
    for (int i = 0; i < LEAD_BATCH; i++) l[i] = k0 + i < K0 ? row[k0 + i] : 0.0;
#pragma unroll
    for (int i = 0; i < LEAD_BATCH; i++) {
      const int k = k0 + i;
      if (k >= K0) break;
      const double lk = (lane > k && lane < K0) ? l[i] : 0.0;
#pragma unroll
      for (int v = 0; v < NV; v++) {
        const double yk = readlane(yl[v], k);
        yl[v] = fma(-lk, yk, yl[v]);
        yt[v] = fma(-a21[k], yk, yt[v]);
      }
    }
  }
}

template <int NV>
__device__ __forceinline__ void solve_trailing(double (&yt)[NV], const double (&c)[NT], double dt, int lane) {
  // the trailing block's solves: at step k every lane takes lane k's final value by v_readlane and is updated with
  // its factor entry in column k, unmasked; the value read, lane k's final one, is written into lane k of the record
  // by v_writelane (before the update spoils lane k; the lanes already recorded are spoilt freely), so a step has no
  // compare or select, and the chain from step to step is a readlane and an fma. pin keeps each step's record in its
  // step: left free, the compiler sinks the records to the end and holds every step's value until then
  double rec[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) rec[v] = 0.0;  // lanes past NT keep 0
  // (a step's writelanes come after its fmas: a written scalar must wait a cycle before v_writelane reads it, and a
  // written vector register before v_readlane reads it, so this order needs no wait instructions)
  double yk[NV];
#pragma unroll
  for (int k = 0; k < NT; k++) {  // unit L, trailing block
#pragma unroll
    for (int v = 0; v < NV; v++) yk[v] = readlane(yt[v], k);
#pragma unroll
    for (int v = 0; v < NV; v++)
      if (k + 1 < NT) yt[v] = fma(-c[k], yk[v], yt[v]);
#pragma unroll
    for (int v = 0; v < NV; v++) rec[v] = writelane(rec[v], yk[v], k);
#pragma unroll
    for (int v = 0; v < NV; v++) pin(rec[v], yt[v]);
  }
#pragma unroll
  for (int v = 0; v < NV; v++) yt[v] = 0.0;
#pragma unroll
  for (int k = NT - 1; k >= 0; k--) {  // unit U' = U diag(1 / U_kk), trailing block
#pragma unroll
    for (int v = 0; v < NV; v++) yk[v] = readlane(rec[v], k);
#pragma unroll
    for (int v = 0; v < NV; v++)
      if (k > 0) rec[v] = fma(-c[k], yk[v], rec[v]);
#pragma unroll
    for (int v = 0; v < NV; v++) yt[v] = writelane(yt[v], yk[v], k);
#pragma unroll
    for (int v = 0; v < NV; v++) pin(rec[v], yt[v]);
  }
#pragma unroll
  for (int v = 0; v < NV; v++) yt[v] *= dt;
}

// U of the lead rows, lead columns.
template <int NV>
__device__ __forceinline__ void solve_lead_upper(double (&yl)[NV], double dl, const double* ws, int lane) {
  const double* row = ws + (lane < K0 ? lane : 0) * NS;
#pragma unroll
  for (int k1 = K0; k1 > 0; k1 -= LEAD_BATCH) {
    double u[LEAD_BATCH];
#pragma unroll
    for (int i = 0; i < LEAD_BATCH; i++) u[i] = k1 - 1 - i >= 0 ? row[k1 - 1 - i] : 0.0;
#pragma unroll
    for (int i = 0; i < LEAD_BATCH; i++) {
      const int k = k1 - 1 - i;
      if (k < 0) break;
      const double uk = lane < k ? u[i] : 0.0;
#pragma unroll
      for (int v = 0; v < NV; v++) yl[v] = fma(-uk, readlane(yl[v] * dl, k), yl[v]);
    }
  }
#pragma unroll
  for (int v = 0; v < NV; v++) yl[v] *= dl;
}

template <int NV>
__device__ __forceinline__ void solve_lead_backward(double (&yl)[NV], const double (&yt)[NV], double dl, double* ws,
                                                    int lane) {
  if constexpr (K0 > 0 && K0 <= SMALL_LEAD) {
    // U of the lead rows, trailing columns: lane t's share of each lead row, summed over the lanes
    double sum[K0 > 0 ? K0 * NV : 1];
#pragma unroll
    for (int i = 0; i < K0; i++) {
      const double a = NT == WAVE || lane < NT ? ws[i * NS + K0 + lane] : 0.0;
#pragma unroll
      for (int v = 0; v < NV; v++) sum[i * NV + v] = a * yt[v];
    }
    wave_sums(sum);
#pragma unroll
    for (int i = 0; i < K0; i++) {
#pragma unroll
      for (int v = 0; v < NV; v++) yl[v] = lane == i ? yl[v] - sum[i * NV + v] : yl[v];
    }
    solve_lead_upper(yl, dl, ws, lane);
  } else if (K0 > 0) {
    // U of the lead rows, trailing columns: the trailing solution through LDS (the union region is free between
    // the right-hand sides), a batch of columns at a time
    double* xv = ws + L_UNION;
    wave_sync();
#pragma unroll
    for (int v = 0; v < NV; v++)
      if (lane < NT) xv[v * NT + lane] = yt[v];
    wave_sync();
    if (lane < K0) {
#pragma unroll 1
      for (int t0 = 0; t0 < NT; t0 += STREAM_BATCH) {
        double a[STREAM_BATCH];
#pragma unroll
        for (int i = 0; i < STREAM_BATCH; i++) a[i] = t0 + i < NT ? ws[lane * NS + K0 + t0 + i] : 0.0;
#pragma unroll
        for (int v = 0; v < NV; v++) {
#pragma unroll
          for (int i = 0; i < STREAM_BATCH; i++)
            if (t0 + i < NT) yl[v] = fma(-a[i], xv[v * NT + t0 + i], yl[v]);
        }
      }
    }
    wave_sync();
    solve_lead_upper(yl, dl, ws, lane);
  }
}

// The trailing solves by blocks of 16 rows, one row of lanes each, for a full trailing block (NT == WAVE) whose c has 0
// on the diagonal. Within a block, lane k's value reaches its row of lanes by DPP inside the fma, and the exec mask
// keeps the lanes already final (their c entries belong to the other triangle); a finished block reaches the other
// rows of lanes through LDS, and its 16 updates there take it by DPP too. An entry takes its updates in the order of
// solve_trailing, so the bits are the same. A step costs 3 issue slots for one vector and 3 for two (an exec shift, an
// fma each, a wait), an update of the other rows one, where a step by v_readlane and v_writelane takes 7 and 11.
// Cycles of one wavefront (NCHO, the lead rows' part included): one vector 5.7k -> 4.1k, two 9.7k -> 5.9k; on
// SNCHO, whose 27 lead columns are now read ahead of their steps, 13.6k -> 8.6k and 20.9k -> 13.5k.
// (DPP reads a register two wait states after a vector instruction wrote it: the other vector's fma and the exec shift,
// or s_nop; the blocks' first and last instructions keep the same distance from the compiler's.)
#define MXC_FWD "s_lshl_b64 exec, exec, 1\n\t"
#define MXC_BWD "s_lshr_b64 exec, exec, 1\n\t"
#define MXC_DPP(Y, X, K, ROWS) "v_fmac_f64_dpp %[" Y "], %[" X "], -%[c" #K "] row_newbcast:" #K " row_mask:" ROWS " bank_mask:0xf\n\t"
#define MXC_ST1(MOVE, K, ROWS) MOVE "s_nop 0\n\t" MXC_DPP("y", "y", K, ROWS)
#define MXC_ST2(MOVE, K, ROWS) MOVE MXC_DPP("y", "y", K, ROWS) MXC_DPP("z", "z", K, ROWS)
#define MXC_UP1(MOVE, K, ROWS) MXC_DPP("y", "p", K, ROWS)
#define MXC_UP2(MOVE, K, ROWS) MXC_DPP("y", "p", K, ROWS) MXC_DPP("z", "q", K, ROWS)
#define MXC_ASC(S, M, R)                                                                                        \
  S("", 0, R) S(M, 1, R) S(M, 2, R) S(M, 3, R) S(M, 4, R) S(M, 5, R) S(M, 6, R) S(M, 7, R) S(M, 8, R) S(M, 9, R) \
  S(M, 10, R) S(M, 11, R) S(M, 12, R) S(M, 13, R) S(M, 14, R)
#define MXC_DESC(S, M, R)                                                                                         \
  S("", 15, R) S(M, 14, R) S(M, 13, R) S(M, 12, R) S(M, 11, R) S(M, 10, R) S(M, 9, R) S(M, 8, R) S(M, 7, R) S(M, 6, R) \
  S(M, 5, R) S(M, 4, R) S(M, 3, R) S(M, 2, R) S(M, 1, R)
#define MXC_COLUMNS                                                                                               \
  [c0] "v"(c[0]), [c1] "v"(c[1]), [c2] "v"(c[2]), [c3] "v"(c[3]), [c4] "v"(c[4]), [c5] "v"(c[5]), [c6] "v"(c[6]),  \
      [c7] "v"(c[7]), [c8] "v"(c[8]), [c9] "v"(c[9]), [c10] "v"(c[10]), [c11] "v"(c[11]), [c12] "v"(c[12]),        \
      [c13] "v"(c[13]), [c14] "v"(c[14]), [c15] "v"(c[15])
// a block's own steps: exec shifted to its lanes (SHIFT), then one place a step
#define MXC_OWN(ST, ORDER, MOVE, SHIFT, ROWS, ...)                                                                 \
  asm volatile("s_mov_b64 %[e], exec\n\t" SHIFT "\n\ts_nop 1\n\t" ORDER(ST, MOVE, ROWS) "s_mov_b64 exec, %[e]\n\ts_nop 1" \
               : __VA_ARGS__, [e] "=&s"(e)                                                                         \
               : MXC_COLUMNS                                                                                      \
               : "scc")
#define MXC_OTHERS(UP, ORDER, LAST, ROWS, OUT, ...) \
  asm volatile("s_nop 1\n\t" ORDER(UP, "", ROWS) UP("", LAST, ROWS) "s_nop 1" : OUT : __VA_ARGS__, MXC_COLUMNS)

template <int B, bool UP>
__device__ __forceinline__ void block_own(double (&yt)[1], const double* c) {
  u64 e;
#define MXC_OWN1(ORDER, MOVE, SHIFT, ROWS) MXC_OWN(MXC_ST1, ORDER, MOVE, SHIFT, ROWS, [y] "+&v"(yt[0]))
  if constexpr (!UP) {
    if constexpr (B == 0) MXC_OWN1(MXC_ASC, MXC_FWD, "s_nop 0", "0x1");
    if constexpr (B == 1) MXC_OWN1(MXC_ASC, MXC_FWD, "s_lshl_b64 exec, exec, 16", "0x2");
    if constexpr (B == 2) MXC_OWN1(MXC_ASC, MXC_FWD, "s_lshl_b64 exec, exec, 32", "0x4");
    if constexpr (B == 3) MXC_OWN1(MXC_ASC, MXC_FWD, "s_lshl_b64 exec, exec, 48", "0x8");
  } else {
    if constexpr (B == 0) MXC_OWN1(MXC_DESC, MXC_BWD, "s_lshr_b64 exec, exec, 48", "0x1");
    if constexpr (B == 1) MXC_OWN1(MXC_DESC, MXC_BWD, "s_lshr_b64 exec, exec, 32", "0x2");
    if constexpr (B == 2) MXC_OWN1(MXC_DESC, MXC_BWD, "s_lshr_b64 exec, exec, 16", "0x4");
    if constexpr (B == 3) MXC_OWN1(MXC_DESC, MXC_BWD, "s_nop 0", "0x8");
  }
}
template <int B, bool UP>
__device__ __forceinline__ void block_own(double (&yt)[2], const double* c) {
  u64 e;
#define MXC_OWN2(ORDER, MOVE, SHIFT, ROWS) MXC_OWN(MXC_ST2, ORDER, MOVE, SHIFT, ROWS, [y] "+&v"(yt[0]), [z] "+&v"(yt[1]))
  if constexpr (!UP) {
    if constexpr (B == 0) MXC_OWN2(MXC_ASC, MXC_FWD, "s_nop 0", "0x1");
    if constexpr (B == 1) MXC_OWN2(MXC_ASC, MXC_FWD, "s_lshl_b64 exec, exec, 16", "0x2");
    if constexpr (B == 2) MXC_OWN2(MXC_ASC, MXC_FWD, "s_lshl_b64 exec, exec, 32", "0x4");
    if constexpr (B == 3) MXC_OWN2(MXC_ASC, MXC_FWD, "s_lshl_b64 exec, exec, 48", "0x8");
  } else {
    if constexpr (B == 0) MXC_OWN2(MXC_DESC, MXC_BWD, "s_lshr_b64 exec, exec, 48", "0x1");
    if constexpr (B == 1) MXC_OWN2(MXC_DESC, MXC_BWD, "s_lshr_b64 exec, exec, 32", "0x2");
    if constexpr (B == 2) MXC_OWN2(MXC_DESC, MXC_BWD, "s_lshr_b64 exec, exec, 16", "0x4");
    if constexpr (B == 3) MXC_OWN2(MXC_DESC, MXC_BWD, "s_nop 0", "0x8");
  }
}

template <int B, bool UP>
__device__ __forceinline__ void block_others(double (&yt)[1], const double (&p)[1], const double* c) {
#define MXC_OTHERS1(ORDER, LAST, ROWS) MXC_OTHERS(MXC_UP1, ORDER, LAST, ROWS, [y] "+&v"(yt[0]), [p] "v"(p[0]))
  if constexpr (!UP) {
    if constexpr (B == 0) MXC_OTHERS1(MXC_ASC, 15, "0xe");
    if constexpr (B == 1) MXC_OTHERS1(MXC_ASC, 15, "0xc");
    if constexpr (B == 2) MXC_OTHERS1(MXC_ASC, 15, "0x8");
  } else {
    if constexpr (B == 3) MXC_OTHERS1(MXC_DESC, 0, "0x7");
    if constexpr (B == 2) MXC_OTHERS1(MXC_DESC, 0, "0x3");
    if constexpr (B == 1) MXC_OTHERS1(MXC_DESC, 0, "0x1");
  }
}
#define MXC_PAIR [y] "+&v"(yt[0]), [z] "+&v"(yt[1])
template <int B, bool UP>
__device__ __forceinline__ void block_others(double (&yt)[2], const double (&p)[2], const double* c) {
#define MXC_OTHERS2(ORDER, LAST, ROWS) \
  asm volatile("s_nop 1\n\t" ORDER(MXC_UP2, "", ROWS) MXC_UP2("", LAST, ROWS) "s_nop 1" \
               : MXC_PAIR : [p] "v"(p[0]), [q] "v"(p[1]), MXC_COLUMNS)
  if constexpr (!UP) {
    if constexpr (B == 0) MXC_OTHERS2(MXC_ASC, 15, "0xe");
    if constexpr (B == 1) MXC_OTHERS2(MXC_ASC, 15, "0xc");
    if constexpr (B == 2) MXC_OTHERS2(MXC_ASC, 15, "0x8");
  } else {
    if constexpr (B == 3) MXC_OTHERS2(MXC_DESC, 0, "0x7");
    if constexpr (B == 2) MXC_OTHERS2(MXC_DESC, 0, "0x3");
    if constexpr (B == 1) MXC_OTHERS2(MXC_DESC, 0, "0x1");
  }
}

template <int B, bool UP, int NV>
__device__ __forceinline__ void block_solve(double (&yt)[NV], const double (&c)[NT], double* xw, int lane) {
  block_own<B, UP>(yt, c + 16 * B);
  if constexpr (UP ? B > 0 : B < 3) {
    double p[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) xw[v * WAVE + lane] = yt[v];
    wave_sync();
#pragma unroll
    for (int v = 0; v < NV; v++) p[v] = xw[v * WAVE + 16 * B + (lane & 15)];
    wave_sync();
    block_others<B, UP>(yt, p, c + 16 * B);
  }
}

template <int NV>
__device__ __forceinline__ void solve_blocks(double (&yt)[NV], const double (&c)[NT], double dt, double* ws, int lane) {
  double* xw = ws + L_UNION;  // free between the right-hand sides
  block_solve<0, false>(yt, c, xw, lane);
  block_solve<1, false>(yt, c, xw, lane);
  block_solve<2, false>(yt, c, xw, lane);
  block_solve<3, false>(yt, c, xw, lane);
  block_solve<3, true>(yt, c, xw, lane);
  block_solve<2, true>(yt, c, xw, lane);
  block_solve<1, true>(yt, c, xw, lane);
  block_solve<0, true>(yt, c, xw, lane);
#pragma unroll
  for (int v = 0; v < NV; v++) yt[v] *= dt;
}

constexpr bool BLOCK_SOLVES = LU_2D && NT == WAVE;  // a try's factors then have 0 on c's diagonal (lu_factor)

// BLOCKS: c has 0 on its diagonal (BLOCK_SOLVES)
template <int NV, bool BLOCKS = false>
__device__ __forceinline__ void solve(double (&yl)[NV], double (&yt)[NV], const double (&c)[NT], const LeadRow& a21,
                                      double dl, double dt, double* ws, int lane) {
  lane = opaque_lane(lane);
  ws = opaque_lds(ws);
  solve_lead_forward(yl, yt, a21, ws, lane);
  if constexpr (BLOCKS)
    solve_blocks(yt, c, dt, ws, lane);
  else
    solve_trailing(yt, c, dt, lane);
  if constexpr (K0 > 0) {  // a rounded product here, not contracted into the sums that follow
#pragma unroll
    for (int v = 0; v < NV; v++) pin(yt[v]);
  }
  solve_lead_backward(yl, yt, dl, ws, lane);
}

__device__ __forceinline__ double vsum(double yl, double yt, int lane) {
  return wave_sum((lane < K0 ? yl : 0.0) + (lane < NT ? yt : 0.0));
}

// ---- step control (the reference's step_factor, next_try and try_error: common.cuh:87-133, 568-589) ----

struct Step {
  double h, t, nok, pen, pha;
  bool prej;
};

__device__ __forceinline__ double step_factor(double en, bool ok, bool prej, double pen, double pha, double ha) {
  const bool efin = isfinite(en);
  double fac = efin ? STEP_SAFETY / cbrt(fmax(en, ERR_FLOOR)) : FAC_NONFINITE;
  fac = fmin(fmax(fac, ok ? FACACC : FACREJ), FACMAX);
  if (!ok && efin && prej && en > 1.0 && pen > 1.0 && pha > ha) {  // secant: err ~ h^pe through the two tries
    const double pe = log(pen / en) / log(pha / ha);
    fac = pe > SECANT_MIN_ORDER ? fmax(pow(SECANT_TARGET / en, 1.0 / fmin(pe, SECANT_MAX_ORDER)), SECMIN) : SECMIN;
  }
  if (!ok) fac = fmin(fac, FAC_AFTER_REJECT);
  return fac;
}

// The try's error (RMS; while no step of the call is accepted, the larger of RMS and max-norm) and its new state y.
__device__ __forceinline__ double try_error(double Nl, double Nt, double K1l, double K1t, double K3l, double K3t,
                                            double K4l, double K4t, double& yl, double& yt, bool first, double rtol,
                                            double atol, int lane, bool& ok) {
  yl = Nl + 2.0 * K1l + K3l + K4l;
  yt = Nt + 2.0 * K1t + K3t + K4t;
  const double ql = K4l / (atol + rtol * fmax(fabs(Nl), fabs(yl)));
  const double qt = K4t / (atol + rtol * fmax(fabs(Nt), fabs(yt)));
  const bool hl = lane < K0, ht = lane < NT;
  const double e2 = wave_sum((hl ? ql * ql : 0.0) + (ht ? qt * qt : 0.0));
  const double em = wave_max(fmax(hl ? fabs(ql) : 0.0, ht ? fabs(qt) : 0.0));
  const bool nn = wave_all((!hl || yl >= -atol) && (!ht || yt >= -atol));
  const double er = sqrt(e2 / NS);
  const double en = (first && isfinite(er)) ? fmax(er, em) : er;
  ok = (en <= 1.0) && nn && isfinite(en);
  return en;
}

// x = N / sum N at the cell's output row (network order); returns the sum.
__device__ __forceinline__ void write_state(double Nl, double Nt, double* __restrict__ out, NetP net,
                                            int lane) {
  const gptr<int> perm = opaque(net)->perm;
  const double s = vsum(Nl, Nt, lane);
  if (lane < K0) out[perm[lane]] = Nl / s;
  if (lane < NT) out[perm[K0 + lane]] = Nt / s;
}
