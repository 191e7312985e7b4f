// Learned warm start of the ALS reductions: a small MLP, trained and run on
// the GPU by the kernels of this file (FP32; products on the matrix cores).
//
// One network serves every mode of the top layer.  Input: a normalised
// factor column x of a state (its n_k entries, zero-padded to nin) and a
// learned embedding e_k of the mode (nemb values); two tanh hidden layers of
// nhid; linear output added to the input, y = x + W3 h2 + b3 (nout = nin).
// The skip connection makes the untrained network (W3 = 0, b3 = 0) the
// plain start F = Psi.  It is trained on pairs
// (x = column r of Psi_t on mode k, t = column r of the ALS-reduced H Psi_t
// on mode k, normalised and sign-aligned with x), which the plain reduced
// H*Q phase produces term by term (the ALS there starts from F = Psi, so
// term r of the result grew out of term r of Psi).  Used as the starting
// factors of that ALS: F_r^k = y / |y|.
//
// Parameters live in one float vector:
//   W1 [nhid][nin+nemb]  b1 [nhid]  W2 [nhid][nhid]  b2 [nhid]
//   W3 [nout][nhid]      b3 [nout]  E  [nmodes][nemb]
// Loss: L = 1/(2N) sum_b |y_b - t_b|^2 over a batch of N columns.

struct MlpDims {
  int nin, nemb, nmodes, nhid, nout;
  __host__ __device__ int nx() const { return nin + nemb; }
  __host__ __device__ long oW1() const { return 0; }
  __host__ __device__ long ob1() const { return (long)nhid * nx(); }
  __host__ __device__ long oW2() const { return ob1() + nhid; }
  __host__ __device__ long ob2() const { return oW2() + (long)nhid * nhid; }
  __host__ __device__ long oW3() const { return ob2() + nhid; }
  __host__ __device__ long ob3() const { return oW3() + (long)nout * nhid; }
  __host__ __device__ long oE() const { return ob3() + nout; }
  __host__ __device__ long np() const { return oE() + (long)nmodes * nemb; }
};

// Products of the network.  A workgroup of four waves forms a 32 x 64 tile of
// sum_k A(i, k) B(j, k) on the FP32 matrix cores (16x16x4), each wave 16 x 32
// of it.  Operands pass through LDS in chunks of 64 k, the next chunk loaded
// into registers while the current one is used.  The tile is small on purpose:
// the matrices have a few thousand rows and a hundred columns, so a call is
// bound by how many workgroups it has (4096 x 128 x 76: 256 of these) and by
// the latency of its two chunks, not by the matrix rate (9 us; a tile of 16 x
// 16 outputs on the vector units took 73).  An LDS row is 68
// floats: the sixteen rows and four k a fragment reads fall into the 64 banks
// once each.
#define MLP_TI 32
#define MLP_TJ 64
#define MLP_TK 64
#define MLP_LD (MLP_TK + 4)

typedef float v4f __attribute__((ext_vector_type(4)));

// An operand X(r, k), r < n: k contiguous (KF, x[r * ld + k]) or r contiguous
// (x[k * ld + r]).
struct MlpOp {
  const float* x;
  long ld;
  int n;
};

// Rows r0 .. r0 + ROWS and k0 .. k0 + 64 of an operand into registers, every
// load unconditional at a clamped address.  Rows past the operand give rows of
// the result that nobody stores; k past the sum are zeroed on the way to LDS.
template <int ROWS, int KF>
__device__ __forceinline__ void mlp_load(float* v, const MlpOp& o, int r0,
                                         int k0, int k1) {
#pragma unroll
  for (int u = 0; u < ROWS * MLP_TK / 256; u++) {
    const int e = u * 256 + (int)threadIdx.x;
    const int r = min(r0 + (KF ? e / MLP_TK : e % ROWS), o.n - 1);
    const int k = min(k0 + (KF ? e % MLP_TK : e / ROWS), k1 - 1);
    v[u] = o.x[KF ? r * o.ld + k : k * o.ld + r];
  }
}

template <int ROWS, int KF>
__device__ __forceinline__ void mlp_store(float* s, const float* v, int nk) {
#pragma unroll
  for (int u = 0; u < ROWS * MLP_TK / 256; u++) {
    const int e = u * 256 + (int)threadIdx.x;
    const int r = KF ? e / MLP_TK : e % ROWS, k = KF ? e % MLP_TK : e / ROWS;
    s[r * MLP_LD + k] = k < nk ? v[u] : 0.0f;
  }
}

// The tile (i0, j0) summed over k0 <= k < k1, in matrix-core layout: c[t][v]
// is row 16 (w & 1) + 4 (lane / 16) + v, column 32 (w >> 1) + 16 t + lane % 16
// for wave w.  With rsum, rs is the sum over k of row tid / 8, in the eight
// threads that share it, of their eighths.
template <int KFA, int KFB>
__device__ __forceinline__ void mlp_tile(v4f c[2], const MlpOp& A,
                                         const MlpOp& B, int i0, int j0, int k0,
                                         int k1, float* As, float* Bs,
                                         bool rsum, float& rs) {
  const int lane = threadIdx.x & 63, lr = lane & 15, lq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wi = 16 * (w & 1), wj = 32 * (w >> 1);
  const bool live = i0 + wi < A.n && j0 + wj < B.n;
  c[0] = c[1] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
  float va[MLP_TI * MLP_TK / 256], vb[MLP_TJ * MLP_TK / 256];
  mlp_load<MLP_TI, KFA>(va, A, i0, k0, k1);
  mlp_load<MLP_TJ, KFB>(vb, B, j0, k0, k1);
  for (; k0 < k1; k0 += MLP_TK) {
    const int nk = min(MLP_TK, k1 - k0);
    mlp_store<MLP_TI, KFA>(As, va, nk);
    mlp_store<MLP_TJ, KFB>(Bs, vb, nk);
    __syncthreads();
    if (k0 + MLP_TK < k1) {
      mlp_load<MLP_TI, KFA>(va, A, i0, k0 + MLP_TK, k1);
      mlp_load<MLP_TJ, KFB>(vb, B, j0, k0 + MLP_TK, k1);
    }
    if (rsum) {
      const float* p = As + (threadIdx.x >> 3) * MLP_LD + (threadIdx.x & 7);
#pragma unroll
      for (int q = 0; q < MLP_TK / 8; q++) rs += p[8 * q];
    }
    if (live) {
      const float* ap = As + (wi + lr) * MLP_LD + lq;
      const float* bp = Bs + (wj + lr) * MLP_LD + lq;
      for (int q0 = 0; q0 < nk; q0 += 16)   // zeros past nk
#pragma unroll
        for (int q = q0; q < q0 + 16; q += 4) {
          const float a = ap[q], b0 = bp[q], b1 = bp[16 * MLP_LD + q];
          c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b0, c[0], 0, 0, 0);
          c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b1, c[1], 0, 0, 0);
        }
    }
    __syncthreads();
  }
}

// What becomes of a product's entries.
struct MlpOut {
  float* C;            // destination (null: not kept), row-major
  long ldc;
  const float* bias;   // added per column, or null
  int tanh;            // tanh of it
  const float* H;      // times 1 - H^2 (the derivative of tanh), or null
  const float* skip;   // the skip connection's input rows, or null
  long lds;
  // loss: target rows T[idx[i]] (null: none), dY = (y - t) scale, and the
  // summed squared error
  const float* T;
  const int* idx;
  float scale;
  float* dY;
  double* sse;
};

// C = out(A B^T) for an M x N product over K.
template <int KFB>
__global__ __launch_bounds__(256) void k_mlp_gemm(MlpOp A, MlpOp B, int K,
                                                   MlpOut o) {
  __shared__ float As[MLP_TI * MLP_LD], Bs[MLP_TJ * MLP_LD];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int i0 = blockIdx.y * MLP_TI, j0 = blockIdx.x * MLP_TJ;
  v4f c[2];
  float rs = 0.0f;
  mlp_tile<1, KFB>(c, A, B, i0, j0, 0, K, As, Bs, false, rs);
  double loc = 0.0;
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int j = j0 + 32 * (w >> 1) + 16 * t + (lane & 15);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int i = i0 + 16 * (w & 1) + 4 * (lane >> 4) + v;
      if (i >= A.n || j >= B.n) continue;
      float s = c[t][v];
      if (o.bias) s += o.bias[j];
      if (o.tanh) s = tanhf(s);
      if (o.H) {
        const float h = o.H[(long)i * o.ldc + j];
        s *= 1.0f - h * h;
      }
      if (o.skip) s += o.skip[(long)i * o.lds + j];
      if (o.C) o.C[(long)i * o.ldc + j] = s;
      if (o.T) {
        const float d = s - o.T[(long)(o.idx ? o.idx[i] : i) * o.ldc + j];
        o.dY[(long)i * o.ldc + j] = d * o.scale;
        loc += (double)d * d;
      }
    }
  }
  if (o.T) {
    // one atomic a workgroup (they all meet in one address)
    __shared__ double ws[4];
    for (int q = 32; q > 0; q >>= 1) loc += __shfl_down(loc, q, 64);
    if (lane == 0) ws[w] = loc;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(o.sse, ws[0] + ws[1] + ws[2] + ws[3]);
  }
}

// Gradients, one part per range of kc batch rows (blockIdx.y), laid out as the
// parameters in part + blockIdx.y * np: the weight gradients sum_b dZ(b, i)
// H(b, j) tile by tile, the bias gradients with the tiles of the first column,
// and in the last workgroup the embedding gradients (the sums of dXe over the
// rows of each mode).  The batch is the long dimension here, so its rows are
// split until the tiles fill the device; k_mlp_gsum adds the parts in order.
// 4096 rows of 60 inputs: this pass (13 us, 672 workgroups) and the sum (9 us)
// take the place of three single-pass products (73 us each, 16 to 64
// workgroups), three column sums by one thread a column (376 us each) and the
// embedding's (789 us).  The squared error goes by one atomic a workgroup
// (one a wave: 16 us for the output layer instead of 12).
struct MlpGrad {
  MlpOp A[3], B[3];     // dZ and H of layers 1 .. 3
  long oW[3], ob[3];    // their places among the parameters
  int t0[4];            // first tile of each layer
  int kc, nb;
  const float* dXe;     // [nb][nemb]
  const int* modes;
  const int* idx;
  int nemb, nmodes;
  long oE, np;
  float* part;
};

__global__ __launch_bounds__(256) void k_mlp_grad(MlpGrad g) {
  __shared__ float As[MLP_TI * MLP_LD], Bs[MLP_TJ * MLP_LD];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int k0 = blockIdx.y * g.kc, k1 = min(k0 + g.kc, g.nb);
  float* part = g.part + (long)blockIdx.y * g.np;
  if ((int)blockIdx.x == g.t0[3]) {
    // thread (rg, e) adds entry e of every ng-th row to its own sums by mode
    // in LDS (at most 256 x 16 of them), which are then added in order of rg
    const int ne = g.nemb, ng = 256 / ne, n = g.nmodes * ne;
    const int e = (int)threadIdx.x % ne, rg = (int)threadIdx.x / ne;
    float* acc = Bs;
    for (int q = threadIdx.x; q < ng * n; q += 256) acc[q] = 0.0f;
    __syncthreads();
    if (rg < ng)
      for (int b0 = k0 + rg; b0 < k1; b0 += 8 * ng) {
        float x[8];
        int md[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int b = min(b0 + u * ng, k1 - 1);
          x[u] = g.dXe[(long)b * ne + e];
          md[u] = g.modes[g.idx ? g.idx[b] : b];
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
          if (b0 + u * ng < k1) acc[rg * n + md[u] * ne + e] += x[u];
      }
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += 256) {
      float s = 0.0f;
      for (int q = 0; q < ng; q++) s += acc[q * n + t];
      part[g.oE + t] = s;
    }
    return;
  }
  int l = 0;
  while (l < 2 && (int)blockIdx.x >= g.t0[l + 1]) l++;
  const MlpOp A = g.A[l], B = g.B[l];
  const int nj = (B.n + MLP_TJ - 1) / MLP_TJ, t = (int)blockIdx.x - g.t0[l];
  const int i0 = t / nj * MLP_TI, j0 = t % nj * MLP_TJ;
  float rs = 0.0f;
  v4f c[2];
  mlp_tile<0, 0>(c, A, B, i0, j0, k0, k1, As, Bs, j0 == 0, rs);
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const int j = j0 + 32 * (w >> 1) + 16 * q + (lane & 15);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int i = i0 + 16 * (w & 1) + 4 * (lane >> 4) + v;
      if (i < A.n && j < B.n) part[g.oW[l] + (long)i * B.n + j] = c[q][v];
    }
  }
  if (j0 == 0) {
    for (int q = 4; q > 0; q >>= 1) rs += __shfl_xor(rs, q, 8);
    const int i = i0 + (int)(threadIdx.x >> 3);
    if ((threadIdx.x & 7) == 0 && i < A.n) part[g.ob[l] + i] = rs;
  }
}

// G = the parts' sum.
__global__ void k_mlp_gsum(long np, int ns, const float* __restrict__ part,
                           float* G) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < np;
       e += (long)gridDim.x * blockDim.x) {
    float s = 0.0f;
    for (int q = 0; q < ns; q++) s += part[(long)q * np + e];
    G[e] = s;
  }
}

// Network input rows: X0[b] = [x_{idx[b]} ; E[mode[idx[b]]]]; clears the
// squared error that the output layer adds up (sse, or null).
__global__ void k_mlp_input(MlpDims m, const float* __restrict__ X,
                            const int* __restrict__ modes,
                            const int* __restrict__ idx, int nb,
                            const float* __restrict__ P, float* X0,
                            double* sse) {
  const int nx = m.nx();
  if (sse && blockIdx.x == 0 && threadIdx.x == 0) *sse = 0.0;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
       e < (long)nb * nx; e += (long)gridDim.x * blockDim.x) {
    const int b = (int)(e / nx), c = (int)(e % nx);
    const int r = idx ? idx[b] : b;
    X0[e] = c < m.nin ? X[(long)r * m.nin + c]
                      : P[m.oE() + (long)modes[r] * m.nemb + (c - m.nin)];
  }
}

// Adam (Kingma & Ba 2015) on every parameter: step t (from 1).
__global__ void k_mlp_adam(long n, float* P, const float* __restrict__ G,
                           float* Mo, float* Vo, float lr, float b1, float b2,
                           float eps, int t) {
  const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n;
       e += (long)gridDim.x * blockDim.x) {
    const float g = G[e];
    const float mo = b1 * Mo[e] + (1.0f - b1) * g;
    const float vo = b2 * Vo[e] + (1.0f - b2) * g * g;
    Mo[e] = mo;
    Vo[e] = vo;
    P[e] -= lr * (mo / c1) / (sqrtf(vo / c2) + eps);
  }
}

// Warm-start inputs from the factor pool: row b = column c0 + b / D on mode
// d = b % D, normalised, as FP32 (zero-padded to nin); modes[b] = d.
__global__ void k_ws_gather(Pool p, int c0, int ncol, int nin, float* X,
                            int* modes) {
  const int D = p.ndof;
  for (long b = blockIdx.x * (long)blockDim.x + threadIdx.x;
       b < (long)ncol * D; b += (long)gridDim.x * blockDim.x) {
    const int c = c0 + (int)(b / D), d = (int)(b % D), n = p.nbas[d];
    const double* f = colp(p, d, c);
    double s = 0.0;
    for (int i = 0; i < n; i++) s += f[i] * f[i];
    const double r = s > 0.0 ? 1.0 / sqrt(s) : 0.0;
    for (int i = 0; i < nin; i++) X[b * nin + i] = i < n ? (float)(f[i] * r) : 0.0f;
    modes[b] = d;
  }
}

// Warm-start factors back into the pool: column c0 + b / D on mode b % D
// becomes y_b / |y_b| (the coefficient is left: the ALS's first mode step
// does not read it).  A prediction of zero norm keeps the old factor.
__global__ void k_ws_scatter(Pool p, int c0, int ncol, int nout,
                             const float* __restrict__ Y) {
  const int D = p.ndof;
  for (long b = blockIdx.x * (long)blockDim.x + threadIdx.x;
       b < (long)ncol * D; b += (long)gridDim.x * blockDim.x) {
    const int c = c0 + (int)(b / D), d = (int)(b % D), n = p.nbas[d];
    double s = 0.0;
    for (int i = 0; i < n; i++) s += (double)Y[b * nout + i] * Y[b * nout + i];
    if (!(s > 0.0) || !isfinite(s)) continue;
    const double r = 1.0 / sqrt(s);
    double* f = colp(p, d, c);
    for (int i = 0; i < n; i++) f[i] = Y[b * nout + i] * r;
  }
}
