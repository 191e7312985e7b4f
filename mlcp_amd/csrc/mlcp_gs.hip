// Gram-Schmidt of one state in one launch (ALS_ORTHO_3, ALSUtils.f90:381-544).
//
// The phase is a chain of nals x D strictly sequential steps per state, each
// far too small to fill the chip, so its time is the time of the hand-overs
// between the workgroups that share a step.  A kernel boundary between
// dependent launches costs 5-6 us (drain, start, first cold loads); a word
// that carries its own step number, written and polled at agent scope,
// reaches a workgroup on another XCD in 0.35-0.5 us.  So one launch runs all
// steps of a state with resident workgroups (one per CU at most, so all of
// the grid is resident at once) that exchange a step's values through such
// words:
//
//   term workgroup l   owns previous state l: refreshes its cross Grams with
//                      the mode updated last, forms PS = prod_{d != k} X_l^d
//                      and the Gram-Schmidt coefficient coef_l = -<Q_l, F>
//                      and publishes the state's part of the right-hand side,
//                      coef_l PS^T (c_l Q_l^k);
//   slice workgroup q  owns SL columns (basis functions) of the mode: forms
//                      the state's own normal matrix and factors it (every
//                      slice workgroup redundantly, so that nobody waits for
//                      the factors) while the terms are formed elsewhere,
//                      sums its columns of the parts, applies the elimination
//                      and publishes its columns of the solution X, not yet
//                      normalised.
//
// Everyone then reads all of X and takes the row norms (the new coefficients)
// itself; the state's renormalisation 1 / |F| is one factor of the whole
// right-hand side and is applied by the slice workgroups.  A step has two
// hand-overs instead of the three of the kernel-per-step form (terms, sum and
// factors, solve), and between them only the reading of 8 R n bytes, two
// small MFMA contractions and the application of ceil(R/4) elimination steps.
//
// What bounds it now: the slices' chain from X to X (24-mode block, rank 32,
// ~24k cycles a step: reading X 2k, Gram and products 5k, the elimination of
// 32 pivots 9k, sums 3k, the two triangular solves 3k, publishing and being
// seen 2k); the terms take half of that beside it, except on large ranks
// (48-mode block), where both take about as long.  Microseconds a step, the
// kernel-per-step form and this one: 23.1 -> 10.3 (24-mode block), 23.9 -> 13.6
// (12-mode, ranks 8-48), 45.6 -> 25.9 (48-mode, ranks 16-64, n = 120),
// 16.5 -> 9.7 (three modes of 24, rank 20).
//
// Words: a double travels as two 8-byte words, each 32 bits of data under the
// 32-bit number of its step; a word is written by one 8-byte store, so a
// reader that sees the number sees the data, and no fence or flag is needed.
// Numbers are never reused (they grow over the whole life of the session), so
// the buffers need no clearing.  Every wait is bounded (a.spin polls); a
// workgroup that gives up raises a.ab, every other one sees it and leaves,
// and the host runs the call again with the kernel-per-step form.

#include <type_traits>

typedef unsigned long long u64;

#define GS_NT 512          // threads of a workgroup (8 waves)
#define GS_SLMAX 2         // most columns of a slice workgroup

struct GsRun {
  Pool p;
  int iv, R, cF, nals;
  const int* col;          // first column and rank per state
  const int* Rl;
  const double* pen;       // penalty of the state
  int nS, SL;              // slice workgroups, columns per slice
  u64* P;                  // [previous state][pstr] parts of the right-hand side
  long pstr;
  u64* X;                  // [2][xstr] solution, by step parity
  long xstr;
  u64* ctrl;               // stop decision of the tolerance form
  double* tsl;             // [previous state][D][slw] product caches
  double* ssl;             // [slice workgroup][D][slw] the state's own
  long slw;
  const unsigned* ebase;   // first step number of the phase
  unsigned eoff;           // ... of the state within it
  int* ab;                 // raised by a wait that ran out
  int spin;                // polls per wait
  int* err;
  int* done;               // tolerance form (null: fixed sweeps)
  double tol2;
};

typedef unsigned v4u __attribute__((ext_vector_type(4)));

// p, which is the same in every lane, in scalar registers.
__device__ __forceinline__ u64* uniform(const u64* p) {
  const u64 v = (u64)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned)v);
  const unsigned hi = __builtin_amdgcn_readfirstlane((int)(unsigned)(v >> 32));
  return (u64*)(((u64)hi << 32) | lo);
}

// A double is the 16 bytes (low half, step, high half, step), so each of its
// two 8-byte words carries its own step number.  All at agent scope (sc1: past
// the per-XCD L2).  Byte offsets from a uniform base.
__device__ __forceinline__ void ll_put(u64* base, unsigned word, double v,
                                       unsigned ep) {
  const u64 b = (u64)__double_as_longlong(v);
  const v4u x = {(unsigned)b, ep, (unsigned)(b >> 32), ep};
  // (wait states that the compiler inserts only around instructions of its
  // own: five between a vector instruction's write of a scalar register and
  // its use as an address, one before the data of a store of more than 8
  // bytes may be overwritten)
  asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc1\n\ts_nop 1"
               :: "v"(word * 8u), "v"(x), "s"(uniform(base)) : "memory");
}

// U such loads in flight together, waited for here.
template <int U>
__device__ __forceinline__ void ll_ld(const u64* base, const unsigned (&o)[U],
                                      v4u (&r)[U]) {
  static_assert(U == 1 || U == 2 || U == 4 || U == 8, "");
  if constexpr (U == 1) {
    asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %1, %2 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(r[0]) : "v"(o[0]), "s"(base) : "memory");
  } else if constexpr (U == 2) {
    asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %2, %4 sc1\n\t"
                 "global_load_dwordx4 %1, %3, %4 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1])
                 : "v"(o[0]), "v"(o[1]), "s"(base) : "memory");
  } else if constexpr (U == 4) {
    asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %4, %8 sc1\n\t"
                 "global_load_dwordx4 %1, %5, %8 sc1\n\t"
                 "global_load_dwordx4 %2, %6, %8 sc1\n\t"
                 "global_load_dwordx4 %3, %7, %8 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
                 : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]), "s"(base)
                 : "memory");
  } else {
    asm volatile("s_nop 4\n\tglobal_load_dwordx4 %0, %8, %16 sc1\n\t"
                 "global_load_dwordx4 %1, %9, %16 sc1\n\t"
                 "global_load_dwordx4 %2, %10, %16 sc1\n\t"
                 "global_load_dwordx4 %3, %11, %16 sc1\n\t"
                 "global_load_dwordx4 %4, %12, %16 sc1\n\t"
                 "global_load_dwordx4 %5, %13, %16 sc1\n\t"
                 "global_load_dwordx4 %6, %14, %16 sc1\n\t"
                 "global_load_dwordx4 %7, %15, %16 sc1\n\ts_waitcnt vmcnt(0)"
                 : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]),
                   "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
                 : "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]), "v"(o[4]),
                   "v"(o[5]), "v"(o[6]), "v"(o[7]), "s"(base)
                 : "memory");
  }
}

// U doubles at base + o[0..U) (words), of step ep, for every lane of the wave
// (all lanes call it, with valid addresses); false if the wait ran out.  After
// a first look at all of them the wait polls one double only: every workgroup
// polling everything it needs takes the bandwidth that the values travel
// through (15.4 -> 11.5 us a step with this and the 16-byte words, 24-mode
// block).
template <int U>
__device__ __forceinline__ bool ll_get(const u64* base, const unsigned (&o)[U],
                                       unsigned ep, double (&v)[U],
                                       const GsRun& a) {
  unsigned ob[U];
  base = uniform(base);
#pragma unroll
  for (int u = 0; u < U; u++) ob[u] = o[u] * 8u;
  v4u r[U];
  for (int t = 0, mode = 0;; t++) {
    if (mode == 1) {
      const unsigned o1[1] = {ob[0]};
      v4u r1[1];
      ll_ld<1>(base, o1, r1);
      if (__all(r1[0].y == ep && r1[0].w == ep)) mode = 2;
    }
    if (mode != 1) {
      ll_ld<U>(base, ob, r);
      bool ok = true;
#pragma unroll
      for (int u = 0; u < U; u++) ok = ok && r[u].y == ep && r[u].w == ep;
      if (__all(ok)) break;
      if (mode == 0 && U > 1) mode = 1;
    }
    if (t >= a.spin) return false;
    if ((t & 255) == 255 &&
        __hip_atomic_load(a.ab, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      return false;
  }
#pragma unroll
  for (int u = 0; u < U; u++)
    v[u] = __hiloint2double((int)r[u].z, (int)r[u].x);
  return true;
}

// start of a phase: step numbers past those of the last phase, flags cleared
__global__ void k_gs_begin(unsigned* ebase, unsigned last, int* ab, int* done,
                           int B) {
  if (threadIdx.x == 0) {
    *ebase += last;
    *ab = 0;
  }
  for (int i = threadIdx.x; i < B; i += blockDim.x) done[i] = 0;
}

// a phase whose waits ran out leaves error bit 16
__global__ void k_gs_end(const int* ab, int* err) {
  if (threadIdx.x == 0 && *ab) atomicOr(err, 16);
}

// Sum over the 64 lanes, the same value in every lane: row shifts and row
// broadcasts inside the vector registers (a shuffle through the LDS unit
// costs ~100 cycles a stage).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS,
                                             0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS,
                                             0xf, true);
  return v + __hiloint2double(hi, lo);
}

__device__ __forceinline__ double lane_value(double v, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                          __builtin_amdgcn_readlane(__double2loint(v), l));
}

__device__ __forceinline__ double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8: lane 15 of each row
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
  return lane_value(v, 63);
}

// 1 / sqrt(x): hardware estimate and two Newton steps.
__device__ __forceinline__ double rsq_nr(double x) {
  double r = __builtin_amdgcn_rsq(x);
#pragma unroll
  for (int i = 0; i < 2; i++) r = fma(r, fma(-0.5 * x * r, r, 0.5), r);
  return r;
}

// v of lane c of this lane's row of 16 lanes (c a constant once unrolled).
// A readlane broadcast of a double costs ~20 cycles, this one register move.
__device__ __forceinline__ double row_bcast(double v, int c) {
#define RB(n) case n: return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + n, 0xf, 0xf, true)
  switch (c) {
    RB(0); RB(1); RB(2); RB(3); RB(4); RB(5); RB(6); RB(7);
    RB(8); RB(9); RB(10); RB(11); RB(12); RB(13); RB(14);
    default: return __builtin_amdgcn_update_dpp(0.0, v, 0x15f, 0xf, 0xf, true);
  }
#undef RB
}

// A = L D L^T, columns 16 PI .. 16 PI + 15, by one wave.  Lane r holds row r
// of the (already updated) panel in po; pd holds the 16 rows of the diagonal
// block, one copy in each row of 16 lanes, from which a column's entries are
// broadcast.  L(r, c), zero for r <= c, goes to Ls[r lst + c], the unscaled
// columns to Us[r 17 + c - 16 PI], 1 / D to dv.  LAST: no rows below the
// diagonal block.  Rows past the rank are rows of the identity.
template <int PI, int RP, bool LAST>
__device__ __forceinline__ void ldl_panel(double (&po)[16], double (&pd)[16],
                                          double* Ls, int lst, double* Us,
                                          double* dv, bool& bad) {
  int lane = TID & 63;
  const int row = min(lane, RP);   // row RP: not read
  double d = row_bcast(pd[0], 0), r = rcp_nr(d), dinv = 0.0;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const int col = 16 * PI + j;
    asm volatile("" : "+v"(lane));   // (the columns' lane masks one at a time)
    bad |= !(d > 0.0);
    const double ld = pd[j] * r, lo = LAST ? ld : po[j] * r;
    dinv = lane == col ? r : dinv;
    // the next pivot first: its reciprocal runs beside the other updates
    if (j < 15) {
      const double b = row_bcast(pd[j], j + 1);
      pd[j + 1] = fma(-ld, b, pd[j + 1]);
      if (!LAST) po[j + 1] = fma(-lo, b, po[j + 1]);
      d = row_bcast(pd[j + 1], j + 1);
      r = rcp_nr(d);
    }
#pragma unroll
    for (int c = j + 2; c < 16; c++) {
      const double b = row_bcast(pd[j], c);
      pd[c] = fma(-ld, b, pd[c]);
      if (!LAST) po[c] = fma(-lo, b, po[c]);
    }
    // (no branch in here: the compiler would put every update off to the
    // block of its first use and keep all the broadcasts until then)
    if (!LAST) Us[row * 17 + j] = po[j];
    Ls[row * lst + col] = lane > col && (!LAST || lane < 16 * PI + 16) ? lo : 0.0;
    // (the scheduler would gather every column's broadcasts at the top)
    __builtin_amdgcn_sched_barrier(0);
  }
  if ((lane >> 4) == PI) dv[lane] = dinv;
}

// Layout of the 8 waves, for row tiles RTM of 16 and 4 NX basis functions:
// the cross Gram (rows j of state l, columns i of the state) is RTM x RTM
// tiles, wave w taking row tile w / 2 and NTT column tiles from (w & 1) NTT
// (waves past the tiles idle); the second contraction's NT column tiles of
// the basis are spread over NTP wave groups, each wave taking every ITG-th
// row tile.
template <int NX, int RTM>
__global__ __launch_bounds__(GS_NT) void k_gs_state(GsRun a) {
  constexpr int NTT = RTM >= 3 ? 2 : 1;
  constexpr int NT = NX / 4, NTP = NT <= 2 ? 2 : (NT <= 4 ? 4 : 8);
  constexpr int ITG = 8 / NTP, NIT = (RTM + ITG - 1) / ITG;
  // LDS strides: XST = 2 (mod 4) with XST / 2 odd, so the 16 rows x 2
  // columns of a half wave's operand reads fall on different banks; BST = 16
  // (mod 32), so two rows of 16 do; the slices' matrices are read a row per
  // lane and have odd strides
  constexpr int KG = NX == 12 ? 6 : 8;   // k-steps whose operands load together
  constexpr int RP = 16 * RTM, XST = 4 * NX + 2, BST = (RTM & 1) ? RP : RP + 16;
  constexpr int AST = RP + 1, LST = RP + 1;
  constexpr int XSZ = RP * XST > (RP + 1) * (LST + 17) ? RP * XST : (RP + 1) * (LST + 17);
  constexpr int BSZ = RP * (BST > AST ? BST : AST);
  extern __shared__ double sm[];
  __shared__ double cc[64], rn[64], dg[64], red[8], s2sh;
  __shared__ int sab, sbad;
  double* Xs = sm;               // X(i, m) at i XST + m
  double* Ls = sm;               // slice: L and a panel of D L^T, over Xs
  double* Us = sm + (RP + 1) * LST;
  double* Bs = sm + XSZ;         // term: PS(j, i) c_j at j BST + i;
                                 // slice: the system matrix at j AST + i
  double* nrm = Bs + BSZ;        // [8][64] partial squares of the rows of X
  double* psum = nrm + GS_NT;    // slice: partial sums of the parts
  double* self = psum + GS_NT;   // slice: the state's own part, [c][64]
  double* Fs = self + 64 * GS_SLMAX;   // slice: F^d, own columns, [d][c][64]
  int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lq = lane >> 4;
  int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  int D = a.p.ndof, R = a.R;
  const int RT = (R + 15) >> 4, nst = a.nals * D;
  const bool slice = (int)blockIdx.x < a.nS;
  int me = slice ? blockIdx.x : blockIdx.x - a.nS;
  int jt = w >> 1, it0 = (w & 1) * NTT;     // this wave's cross tiles
  const bool cw = jt < RTM && it0 < RT;
  const unsigned ep0 = *a.ebase + a.eoff;
  if (tid == 0) {
    sab = __hip_atomic_load(a.ab, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s2sh = 0.0;
    sbad = 0;
  }
  if (tid < 64) cc[tid] = tid < R ? a.p.coef[a.cF + tid] : 0.0;
  __syncthreads();
  if (sab) return;

  // R x n values over the threads without divisions: rows i over 16, 32 or 64
  // lanes (rsh), columns over the rest
  const int rsh = R <= 16 ? 4 : (R <= 32 ? 5 : 6);
  int ti = tid & ((1 << rsh) - 1), tm = tid >> rsh;
  const int tms = GS_NT >> rsh;
  // Values every step derives its addresses from, made opaque at the start
  // of a step: hoisted out of the step loop, the addresses of all its parts
  // together overflow the register file.
#define GS_OPAQUE()                                                         \
  do {                                                                      \
    asm volatile("" : "+v"(tid), "+v"(lane), "+v"(lr), "+v"(lq), "+v"(ti),  \
                 "+v"(tm));                                                 \
    asm volatile("" : "+s"(w));                                             \
    asm volatile("" : "+s"(D));                                             \
    asm volatile("" : "+s"(R));                                             \
    asm volatile("" : "+s"(me));                                            \
    asm volatile("" : "+s"(jt));                                            \
    asm volatile("" : "+s"(it0));                                           \
  } while (0)
  // zeroes of Xs past the rank and past the basis (the operands of the
  // contractions run over whole tiles)
  auto pad = [&](int n) __attribute__((always_inline)) {
    const int np = (n + 4 * KG - 1) / (4 * KG) * (4 * KG);
    for (int m = n + w; m < np; m += 8)
      if (lane < R) Xs[lane * XST + m] = 0.0;
    for (int i = R + w; i < 16 * RT; i += 8)
      for (int m = lane; m < np; m += 64) Xs[i * XST + m] = 0.0;
  };
  // tile (jt, it0 + q) of <row j, X_i>, rows from registers or (self) from X
  // (column tiles past the rank are formed from whatever Xs holds there and
  // never used: a guard per tile would keep the reads from being batched)
  auto cross = [&](const double (&aq)[NX], auto OWN_, int n, v4d (&acc)[NTT]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NTT; q++) acc[q] = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < NX; k0 += KG)
      if (4 * k0 < n) {   // uniform
        double av[KG], bv[KG][NTT];
#pragma unroll
        for (int b = 0; b < KG; b++) {
          const int mc = 4 * (k0 + b) + lq;
          av[b] = decltype(OWN_)::value ? Xs[(16 * jt + lr) * XST + mc] : aq[k0 + b];
#pragma unroll
          for (int q = 0; q < NTT; q++)
            bv[b][q] = Xs[(16 * min(it0 + q, RTM - 1) + lr) * XST + mc];
        }
#pragma unroll
        for (int b = 0; b < KG; b++)
#pragma unroll
          for (int q = 0; q < NTT; q++) acc[q] = mfma_f64_4(av[b], bv[b][q], acc[q]);
      }
  };
  // rows 16 jt + lr of a factor (columns c0.. of the pool, rank rl) on mode d,
  // repeating the last row and entry past the rank and the basis: what they
  // give is multiplied by zero (c_j past the rank, X past the basis) or not
  // stored
  auto rows_pool = [&](int d, int c0, int rl, double (&aq)[NX]) __attribute__((always_inline)) {
    const int n = a.p.nbas[d], j = 16 * jt + lr;
    const double* f = colp(a.p, d, c0);   // uniform
    const unsigned jo = (unsigned)min(j, rl - 1) * n;
#pragma unroll
    for (int ks = 0; ks < NX; ks++) {
      const int m = 4 * ks + lq;
      aq[ks] = f[jo + (unsigned)min(m, n - 1)];
    }
  };
  // this wave's entries of product cache array d of cache set s
  auto slot = [&](double* base, int s, int d, int q) __attribute__((always_inline)) {
    // (a uniform pointer; the lane's entries are 64 v + lane)
    return base + (((long)s * D + d) * a.slw + (jt * 2 * NTT + it0 + q) * 256);
  };
  double* const sl = slice ? a.ssl : a.tsl;

  // ---- the first step's Grams on every mode, from the factors as they are;
  // the next mode's operands are on their way while one is contracted
  {
    const int r0 = slice ? R : a.Rl[me], c0 = slice ? a.cF : a.col[me];
    const bool on = cw && 16 * jt < r0;
    constexpr int FU = RTM <= 1 ? (NX + 7) / 8 : (RTM == 2 ? NX / 4 : NX / 2);
    double aq[NX], fv[FU];   // FU tms >= 4 NX columns
    auto fetch = [&](int d) __attribute__((always_inline)) {
      const int n = a.p.nbas[d];
      const double* f = colp(a.p, d, a.cF);
#pragma unroll
      for (int u = 0; u < FU; u++)
        fv[u] = f[min(ti, R - 1) * n + min(tm + u * tms, n - 1)];
      if (on) rows_pool(d, c0, r0, aq);
    };
    fetch(0);
    for (int d = 0; d < D; d++) {
      const int n = a.p.nbas[d];
      __syncthreads();   // Xs of the previous mode is read
#pragma unroll
      for (int u = 0; u < FU; u++)
        if (ti < R && tm + u * tms < n) Xs[ti * XST + tm + u * tms] = fv[u];
      pad(n);
      __syncthreads();
      if (on) {
        v4d x[NTT];
        cross(aq, std::false_type(), n, x);
#pragma unroll
        for (int q = 0; q < NTT; q++)
#pragma unroll
          for (int v = 0; v < 4; v++) slot(sl, me, d, q)[64 * v + lane] = x[q][v];
      }
      if (d + 1 < D) fetch(d + 1);
      if (slice) {
        const int m0 = me * a.SL, nc = min(a.SL, n - m0);
        if (w < nc && lane < R)
          Fs[(d * GS_SLMAX + w) * 64 + lane] = Xs[lane * XST + m0 + w];
      }
    }
  }

  // Products of the caches at step k once x = X^{kp} is known: tot =
  // prod_d X^d and ps = prod_{d != k} X^d.  Array d holds X^d where mode d
  // has been updated in this sweep, else the suffix product
  // X^d X^{d+1} ... X^{D-1} of the sweep's start; the prefix product
  // pa = X^0 ... X^{k-1} and the two suffixes of the step stay in registers,
  // so a step reads one array (p1, of mode k + 1, requested ahead) and writes
  // one, whatever the number of modes.
  auto products = [&](int set, int k, const v4d (&x)[NTT], v4d (&pa)[NTT],
                      v4d (&p0)[NTT], const v4d (&p1)[NTT], int rl,
                      v4d (&tot)[NTT], v4d (&ps)[NTT]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NTT; q++) {
      if (k == 0) {
        v4d sv = x[q], s1;
#pragma unroll
        for (int v = 0; v < 4; v++) {
          slot(sl, set, D - 1, q)[64 * v + lane] = sv[v];
          const bool in = 16 * jt + lq + 4 * v < rl && 16 * (it0 + q) + lr < R;
          s1[v] = D == 1 ? (in ? 1.0 : 0.0) : sv[v];
        }
        for (int d1 = D - 2; d1 >= 0; d1 -= 4) {
          v4d xv[4];
#pragma unroll
          for (int u = 0; u < 4; u++)
#pragma unroll
            for (int v = 0; v < 4; v++)
              xv[u][v] = slot(sl, set, max(d1 - u, 0), q)[64 * v + lane];
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const int d = d1 - u;
            if (d >= 0) {
              if (d == 0) s1 = sv;
              sv = sv * xv[u];
#pragma unroll
              for (int v = 0; v < 4; v++) slot(sl, set, d, q)[64 * v + lane] = sv[v];
            }
          }
        }
        tot[q] = sv;
        ps[q] = s1;
        p0[q] = s1;
      } else {
        pa[q] = k == 1 ? x[q] : pa[q] * x[q];
#pragma unroll
        for (int v = 0; v < 4; v++) slot(sl, set, k - 1, q)[64 * v + lane] = x[q][v];
        tot[q] = pa[q] * p0[q];
        ps[q] = k < D - 1 ? pa[q] * p1[q] : pa[q];
        p0[q] = p1[q];
      }
    }
  };
  // array of mode k + 1 for step k (at k = 0 and D - 1 it is not used)
  auto slot_ahead = [&](int set, int k, v4d (&p1)[NTT]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NTT; q++)
#pragma unroll
      for (int v = 0; v < 4; v++)
        p1[q][v] = slot(sl, set, min(k + 1, D - 1), q)[64 * v + lane];
  };
  // step 0 takes X^{D-1} from its array, the others compute it
  auto first_x = [&](int set, v4d (&x)[NTT]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < NTT; q++)
#pragma unroll
      for (int v = 0; v < 4; v++) x[q][v] = slot(sl, set, D - 1, q)[64 * v + lane];
  };
  // X of step s - 1 into Xs, the partial squares of its rows into nrm (all
  // threads; false if the wait ran out)
  auto get_batch = [&](int s, int m0, int n, double& sq, auto U_) __attribute__((always_inline)) {
    constexpr int U = decltype(U_)::value;
    const u64* xb = a.X + (long)((s - 1) & 1) * a.xstr;
    const int ic = min(ti, R - 1);
    unsigned o[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; u++)
      o[u] = 2u * (unsigned)(min(m0 + u * tms, n - 1) * R + ic);
    const bool ok = ll_get<U>(xb, o, ep0 + s, v, a);
    if (ti < R) {
#pragma unroll
      for (int u = 0; u < U; u++)
        if (m0 + u * tms < n) {
          Xs[ti * XST + m0 + u * tms] = v[u];
          sq = fma(v[u], v[u], sq);
        }
    }
    return ok;
  };
  auto get_x = [&](int s, int n) __attribute__((always_inline)) {
    bool ok = true;
    double sq = 0.0;
    if (n <= 2 * tms)
      ok = get_batch(s, tm, n, sq, std::integral_constant<int, 2>());
    else
      for (int m = tm; m - tm < n && ok; m += 4 * tms)
        ok = get_batch(s, m, n, sq, std::integral_constant<int, 4>());
    nrm[tid] = sq;
    pad(n);
    return ok;
  };
  // 1 / |X_i| and the new coefficient |X_i| (every wave for its own rows)
  auto row_norm = [&](int i, double& c) __attribute__((always_inline)) {
    const int ic = min(i, R - 1);
    double t = 0.0;
    for (int g0 = 0; g0 < tms; g0 += 8) {
      double v[8];
#pragma unroll
      for (int g = 0; g < 8; g++) v[g] = nrm[((g0 + g) << rsh) + ic];
      t += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    const double r = rsq_nr(t);
    c = i < R ? t * r : 0.0;
    return i < R && t > 0.0 ? r : 0.0;
  };
  auto give_up = [&]() __attribute__((always_inline)) {
    if (lane == 0) {
      sab = 1;
      __hip_atomic_store(a.ab, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };

  if (!slice) {
    // ---------------------------------------------------- term workgroup
    const int mt = w % NTP, itg = w / NTP;   // this wave's tiles of P
    const int rl = a.Rl[me], c0 = a.col[me];
    const bool cwt = cw && 16 * jt < rl;
    double aq[NX], qk[4 * RTM], cl[4];
    v4d pa[NTT], p0[NTT], p1[NTT];   // (set by the first step)
    // Operands of a step, requested ahead: the state's factor on mode k as
    // the second contraction takes it, and a product cache.
    auto ahead = [&](int k) __attribute__((always_inline)) {
      const int n = a.p.nbas[k];
      const double* fk = colp(a.p, k, c0);   // uniform
      const unsigned mc = (unsigned)min(16 * mt + lr, n - 1);
#pragma unroll
      for (int ks = 0; ks < 4 * RTM; ks++)
        qk[ks] = fk[(unsigned)min(4 * ks + lq, rl - 1) * n + mc];
      if (cwt) slot_ahead(me, k, p1);
    };
    ahead(0);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int j = 16 * jt + lq + 4 * v;
      cl[v] = ld_or0(a.p.coef + c0 + min(j, rl - 1), j < rl);
    }
    u64* const pt = a.P + (long)me * a.pstr;
    for (int s = 0, k = 0; s < nst; s++, k = k + 1 == D ? 0 : k + 1) {
      GS_OPAQUE();
      const int kp = k == 0 ? D - 1 : k - 1, kn = k + 1 == D ? 0 : k + 1;
      const int n = a.p.nbas[k], np = a.p.nbas[kp];
      if (s > 0) {
        bool ok = true;
        if (a.done && kp == 0 && s > D) {
          // the step before tested the tolerance: stop or go on
          const unsigned o[1] = {0u};
          double c[1];
          ok = ll_get<1>(a.ctrl, o, ep0 + s, c, a);
          if (ok && c[0] != 0.0) return;   // the same word for every thread
        }
        if (ok) ok = get_x(s, np);
        if (!ok) give_up();
      }
      __syncthreads();
      if (sab) return;
      double cs = 0.0;
      if (cwt) {
        v4d x[NTT], tot[NTT], ps[NTT];
        double ci[NTT];
        if (s > 0) {
          double ri[NTT];
#pragma unroll
          for (int q = 0; q < NTT; q++)
            ri[q] = row_norm(16 * (it0 + q) + lr, ci[q]);
          cross(aq, std::false_type(), np, x);
#pragma unroll
          for (int q = 0; q < NTT; q++) x[q] = x[q] * ri[q];
        } else {
          first_x(me, x);
#pragma unroll
          for (int q = 0; q < NTT; q++) ci[q] = cc[min(16 * (it0 + q) + lr, 63)];
        }
        // the registers of the rows are free: those of mode k, which the next
        // step contracts with the X that this one leads to
        rows_pool(k, c0, rl, aq);
        products(me, k, x, pa, p0, p1, rl, tot, ps);
#pragma unroll
        for (int q = 0; q < NTT; q++) {
          const int i = 16 * (it0 + q) + lr;
#pragma unroll
          for (int v = 0; v < 4; v++) {
            cs = fma(i < R ? tot[q][v] : 0.0, cl[v] * ci[q], cs);
            if (RTM != 3 || i < RP)
              Bs[(16 * jt + lq + 4 * v) * BST + i] = ps[q][v] * cl[v];
          }
        }
      }
      cs = wave_sum(cs);
      if (lane == 0) red[w] = cs;
      __syncthreads();
      double cf = 0.0;
#pragma unroll
      for (int g = 0; g < 8; g++) cf += red[g];
      v4d acc[NIT];
#pragma unroll
      for (int q = 0; q < NIT; q++) acc[q] = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int k0 = 0; k0 < 4 * RTM; k0 += 4)
        if (4 * k0 < rl) {   // uniform
          double av[4][NIT];
#pragma unroll
          for (int b = 0; b < 4; b++)
#pragma unroll
            for (int q = 0; q < NIT; q++)
              av[b][q] = Bs[(4 * (k0 + b) + lq) * BST + 16 * min(itg + q * ITG, RTM - 1) + lr];
#pragma unroll
          for (int b = 0; b < 4; b++)
#pragma unroll
            for (int q = 0; q < NIT; q++) acc[q] = mfma_f64_4(qk[k0 + b], av[b][q], acc[q]);
        }
      // the next operands are requested before the words are stored: a load
      // behind the stores would wait for their acknowledgement
      ahead(kn);
#pragma unroll
      for (int q = 0; q < NIT; q++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          // element v of the tile (the factor's column first): basis function
          // 16 mt + lq + 4 v, row lr, so 16 lanes store 256 bytes in a row
          const int m = 16 * mt + lq + 4 * v, i = 16 * (itg + q * ITG) + lr;
          if (m < n && i < R)
            ll_put(pt, 2 * (m * R + i), -cf * acc[q][v], ep0 + s + 1);
        }
      if (tid == 0 && a.done) ll_put(pt, a.pstr - 2, cf * cf, ep0 + s + 1);
    }
    return;
  }

  // ------------------------------------------------------ slice workgroup
  // the state as it is left: this slice's columns of every factor, and the
  // coefficients.  (Only here: a workgroup without columns in the first modes
  // may still be reading the old factors in the first steps.)
  auto finish = [&](double rs) __attribute__((always_inline)) {
    for (int d = 0; d < D; d++) {
      const int m0 = me * a.SL, nc = min(a.SL, a.p.nbas[d] - m0);
      if (w < nc && lane < R)
        colp(a.p, d, a.cF + lane)[m0 + w] = Fs[(d * GS_SLMAX + w) * 64 + lane];
    }
    if (me == 0 && tid < R) a.p.coef[a.cF + tid] = cc[tid] * rs;
  };
  const int m0 = me * a.SL;
  const double pen = *a.pen;
  v4d pa[NTT], p0[NTT];   // (set by the first step)
  for (int s = 0, k = 0; s <= nst; s++, k = k + 1 == D ? 0 : k + 1) {
    GS_OPAQUE();
    const bool fin = s == nst;
    const int kp = k == 0 ? D - 1 : k - 1, n = a.p.nbas[k];
    // columns of this slice, and the threads an element of its sums
    const int nc = max(0, min(a.SL, n - m0)), two = nc > 1 ? 1 : 0;
    const bool tile = cw && jt < RT;
    double cs = 0.0;
    {
      v4d p1[NTT], x[NTT], tot[NTT], ps[NTT];
      if (tile) slot_ahead(me, k, p1);
      if (s > 0) {
        __syncthreads();   // L of the last step, over Xs, is read
        if (!get_x(s, a.p.nbas[kp])) give_up();
      }
      __syncthreads();
      if (sab) return;
      __builtin_amdgcn_sched_barrier(0);
      if (s > 0) {
        const int np = a.p.nbas[kp];
        // wave 7 the row norms, which are the new coefficients
        if (w == 7) {
          double c;
          rn[lane] = row_norm(lane, c);
          cc[lane] = c;
          if (lane < R && (c != c || c == 0.0)) atomicOr(a.err, 1);
        }
        if (tile) {
          const double none[NX] = {};
          cross(none, std::true_type(), np, x);
        }
        __syncthreads();
        // the updated factor's own columns, normalised
        const int q0 = 7 - w;
        if (q0 < min(a.SL, np - m0) && lane < R)
          Fs[(kp * GS_SLMAX + q0) * 64 + lane] = Xs[lane * XST + m0 + q0] * rn[lane];
        if (tile) {
#pragma unroll
          for (int v = 0; v < 4; v++) {
            const int j = 16 * jt + lq + 4 * v;
            const double r = rn[j], c = cc[j];
#pragma unroll
            for (int q = 0; q < NTT; q++) {
              const int i = min(16 * (it0 + q) + lr, 63);
              x[q][v] *= r * rn[i];
              tot[q][v] = c * cc[i];   // for the norm below
            }
          }
        }
      }
      if (tile) {
        if (s == 0) first_x(me, x);
        v4d wt[NTT];
#pragma unroll
        for (int q = 0; q < NTT; q++) wt[q] = tot[q];
        if (fin) {
#pragma unroll
          for (int q = 0; q < NTT; q++) {
            tot[q] = D > 1 ? pa[q] * x[q] : x[q];
            ps[q] = tot[q];
          }
        } else {
          products(me, k, x, pa, p0, p1, R, tot, ps);
        }
#pragma unroll
        for (int q = 0; q < NTT; q++) {
          const int i = 16 * (it0 + q) + lr;
#pragma unroll
          for (int v = 0; v < 4; v++) {
            // (the penalty on the diagonal, the identity past the rank)
            const int j = 16 * jt + lq + 4 * v;
            const bool in = i < R && j < R;
            if (s > 0) cs = fma(in ? tot[q][v] : 0.0, wt[q][v], cs);
            if (RTM != 3 || i < RP)
              Bs[j * AST + i] = (in ? ps[q][v] : 0.0) +
                                (i == j ? (in ? pen : 1.0) : 0.0);
            if (i == j) dg[i] = in ? ps[q][v] : 0.0;
          }
        }
      }
    }
    cs = wave_sum(cs);
    if (lane == 0) red[w] = cs;
    __syncthreads();
    double nn = 0.0;
#pragma unroll
    for (int g = 0; g < 8; g++) nn += red[g];
    const double rs = s > 0 ? 1.0 / sqrt(fabs(nn)) : 1.0;
    if (fin) {
      finish(rs);
      return;
    }
    // L D L^T of BB + pen I: wave 0 a panel of 16 columns at a time, all waves
    // the trailing tiles on the matrix cores; meanwhile waves 6 and 7 form
    // the state's own part, sum_j BB(j, i) c_j F_j^k(m).  Rows past the rank
    // are the identity's.
    auto panel = [&](auto PI_) __attribute__((always_inline)) {
      constexpr int PI = decltype(PI_)::value;
      if (PI < RTM && PI < RT) {   // uniform
        const int rd = 16 * PI + lr;   // this lane's row of the diagonal block
        if (w == 0 && nc > 0) {
          double po[16], pd[16];
          bool bad = false;
#pragma unroll
          for (int c = 0; c < 16; c++) {
            pd[c] = Bs[rd * AST + 16 * PI + c];
            po[c] = Bs[min(lane, 16 * RT - 1) * AST + 16 * PI + c];
          }
          if (PI + 1 < RT) {   // uniform
            ldl_panel<PI, RP, false>(po, pd, Ls, LST, Us, nrm, bad);
          } else {
            ldl_panel<PI, RP, true>(po, pd, Ls, LST, Us, nrm, bad);
          }
          if (bad && lane == 0) sbad = 1;
        } else if (PI == 0 && w >= 6 && 7 - w < nc && lane < R) {
          const int c = 7 - w;
          const double* fk = Fs + (k * GS_SLMAX + c) * 64;
          double t[4] = {0.0, 0.0, 0.0, 0.0};
          int j = 0;
          for (; j + 3 < R; j += 4)
#pragma unroll
            for (int u = 0; u < 4; u++)
              t[u] = fma(Bs[(j + u) * AST + lane], cc[j + u] * fk[j + u], t[u]);
          for (; j < R; j++) t[0] = fma(Bs[j * AST + lane], cc[j] * fk[j], t[0]);
          // (without the penalty)
          t[1] = fma(dg[lane] - Bs[lane * AST + lane], cc[lane] * fk[lane], t[1]);
          self[c * 64 + lane] = (t[0] + t[1]) + (t[2] + t[3]);
        }
        if (PI + 1 < RT) {   // uniform
          __syncthreads();
          // trailing tiles (rt, ct), rt >= ct > PI: tile number w
          const int nt = RT - PI - 1;
          int ct = 0, rem = w;
          while (ct < nt && rem >= nt - ct) { rem -= nt - ct; ct++; }
          if (ct < nt && nc > 0) {
            const int rt = PI + 1 + ct + rem;
            ct += PI + 1;
            v4d acc;
            double av[4], bv[4];
#pragma unroll
            for (int v = 0; v < 4; v++)
              acc[v] = Bs[(16 * rt + lq + 4 * v) * AST + 16 * ct + lr];
#pragma unroll
            for (int b = 0; b < 4; b++) {
              av[b] = Ls[(16 * rt + lr) * LST + 16 * PI + 4 * b + lq];
              bv[b] = -Us[(16 * ct + lr) * 17 + 4 * b + lq];
            }
#pragma unroll
            for (int b = 0; b < 4; b++) acc = mfma_f64_4(av[b], bv[b], acc);
#pragma unroll
            for (int v = 0; v < 4; v++)
              Bs[(16 * rt + lq + 4 * v) * AST + 16 * ct + lr] = acc[v];
          }
          __syncthreads();
        }
      }
    };
    panel(std::integral_constant<int, 0>());
    panel(std::integral_constant<int, 1>());
    panel(std::integral_constant<int, 2>());
    panel(std::integral_constant<int, 3>());
    const bool chk = a.done && k == 0 && s > 0;
    {
      // sum of the parts over this slice: thread (row ti, column c, group g)
      // takes the parts g, g + ngr, ... (with two columns, even waves the
      // first and odd waves the second)
      const int c = two ? w & 1 : 0, ngr = two ? (4 << (6 - rsh)) : tms;
      const int g = two ? ((w >> 1) << (6 - rsh)) + (lane >> rsh) : tm;
      bool ok = true;
      if (nc > 0) {   // uniform
        constexpr int U = 8;
        const u64* pe = a.P + 2 * (long)m0 * R;   // uniform
        const unsigned eo = 2u * (unsigned)(c * R + min(ti, R - 1));
        const unsigned pst = (unsigned)a.pstr;
        double sum[4] = {0.0, 0.0, 0.0, 0.0};
        for (int c0 = 0; c0 < a.iv && ok; c0 += U * ngr) {
          unsigned o[U];
          double v[U];
#pragma unroll
          for (int u = 0; u < U; u++)
            o[u] = eo + (unsigned)min(g + c0 + u * ngr, a.iv - 1) * pst;
          ok = ll_get<U>(pe, o, ep0 + s + 1, v, a);
#pragma unroll
          for (int u = 0; u < U; u++)
            if (g + c0 + u * ngr < a.iv) sum[u & 3] += v[u];
        }
        psum[((c * ngr + g) << rsh) + ti] = (sum[0] + sum[1]) + (sum[2] + sum[3]);
      }
      if (chk && w == 7) {
        double t = 0.0;
        for (int c0 = 0; c0 < a.iv && ok; c0 += 64) {
          const unsigned o[1] = {(unsigned)min(c0 + lane, a.iv - 1) * (unsigned)a.pstr};
          double v[1];
          ok = ll_get<1>(a.P + a.pstr - 2, o, ep0 + s + 1, v, a);
          if (c0 + lane < a.iv) t += v[0];
        }
        t = wave_sum(t);
        if (lane == 0) s2sh = t;
      }
      if (!ok) give_up();
    }
    __syncthreads();
    if (sab) return;
    if (chk) {
      // the state's component along the previous (normalised) states,
      // sqrt(sum_l <Q_l, F>^2) with |F| = 1, is within the tolerance: stop
      const bool stop = rs * rs * s2sh <= a.tol2;
      if (me == 0 && tid == 0) ll_put(a.ctrl, 0, stop ? 1.0 : 0.0, ep0 + s + 1);
      if (stop) {
        finish(rs);
        if (me == 0 && tid == 0) a.done[a.iv] = s / D;
        return;
      }
    }
    if (7 - w < nc) {
      // column m0 + c, lane = row: L y = b, then L^T x = D^-1 y, 16 unknowns a
      // block, one copy of them in each row of 16 lanes
      const int c = 7 - w;
      if (sbad && lane == 0) atomicOr(a.err, 2);
      const int ngr = two ? (4 << (6 - rsh)) : tms, i = min(lane, R - 1);
      const int row = min(lane, RP - 1);
      double y = self[c * 64 + i];
      for (int g0 = 0; g0 < ngr; g0 += 4) {
        double v[4];
#pragma unroll
        for (int g = 0; g < 4; g++) v[g] = psum[((c * ngr + g0 + g) << rsh) + i];
        y += (v[0] + v[1]) + (v[2] + v[3]);
      }
      y = lane < R ? y * rs : 0.0;
      const double di = nrm[row];
#pragma unroll
      for (int PI = 0; PI < RTM; PI++)
        if (PI < RT) {   // uniform
          double ld[16], lo[16];
#pragma unroll
          for (int j = 0; j < 16; j++) {
            ld[j] = Ls[(16 * PI + lr) * LST + 16 * PI + j];
            lo[j] = Ls[row * LST + 16 * PI + j];
          }
          double yd = __shfl(y, 16 * PI + lr, 64);
#pragma unroll
          for (int j = 0; j < 16; j++) {
            const double b = row_bcast(yd, j);
            yd = fma(-ld[j], b, yd);
            y = fma(-lo[j], b, y);
          }
          __builtin_amdgcn_sched_barrier(0);   // one block's L at a time
        }
      y = lane < R ? y * di : 0.0;
#pragma unroll
      for (int PI = RTM - 1; PI >= 0; PI--)
        if (PI < RT) {   // uniform
          double ld[16], lo[16];
#pragma unroll
          for (int j = 0; j < 16; j++) {
            ld[j] = Ls[(16 * PI + j) * LST + 16 * PI + lr];
            lo[j] = Ls[(16 * PI + j) * LST + row];
          }
          double yd = __shfl(y, 16 * PI + lr, 64);
#pragma unroll
          for (int j = 15; j >= 0; j--) {
            const double b = row_bcast(yd, j);
            yd = fma(-ld[j], b, yd);
            y = fma(-lo[j], b, y);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      u64* xo = a.X + (long)(s & 1) * a.xstr;
      if (lane < R) ll_put(xo, 2 * ((m0 + c) * R + lane), y, ep0 + s + 1);
    }
  }
}
