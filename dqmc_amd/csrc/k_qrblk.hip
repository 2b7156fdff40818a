// Blocked Householder QR on a chain group, and the solve that uses it.
//
// k_qr_pipe (8-column panels, the default) and k_qr_blocked (16) factor A P0 = Q R panel by
// panel (compact WY, Q_p = I - V_p T_p V_p^H, LAPACK zgeqrf/zlarft conventions). P0 is either
// the identity or the pre-pivoting
// order: columns sorted once by decreasing initial norm (ties by index). For the
// column-graded products DQMC stabilises, (B...B U) diag(D), QR with pre-pivoting is
// as stable as column-pivoted QR (Bai, Lee, Li, Xu, "Stable solutions of linear systems
// involving long chain of matrix multiplications", Linear Algebra Appl. 435 (2011)),
// while the workgroups exchange once per panel (k_qr_pipe by flags, k_qr_blocked by a group
// barrier) instead of once per column.
//
// The output uses the layout of k_qrp (columns never move: logical column k lives in
// physical column qr_perm[k]; reflector k below the diagonal of that column, R on and
// above it; qr_tau[k]; D[k] = |Re R_kk|), so k_form_T / k_form_Q form U and T of
// decompose_udt (linalg.jl:20-39) unchanged. The T factors of all panels are kept in
// qr_Tf for k_qr_solve.
//
// Per panel p, with one-panel look-ahead: workgroup 0 applies Q_p^H to panel p+1's columns
// and factors panel p+1 in registers (zlarfg per column, applied to the rest of the panel,
// with the zlarft inner products formed along the way) while the other workgroups apply
// Q_p^H to the columns beyond.
#include "chain.hpp"

namespace dqmc {

constexpr int kQrMaxN = 1024;
constexpr int kQrMaxNb = 16;

typedef double v4d __attribute__((ext_vector_type(4)));
// one v_mfma_f64_16x16x4: c + A B for this lane's A(i, k) = a, B(k, j) = b
__device__ inline v4d mfma4(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
// LDS column stride of the panel V and of LDS-resident column blocks: >= n and 1 mod 16, so
// that the 16 columns a quarter-wave reads at one row (128-bit accesses) fall on 16 different
// groups of four banks
inline int mfma_ld(int nmax) { return nmax + ((17 - (nmax & 15)) & 15); }

__device__ inline cplx shfl_c(cplx v, int src) { return mk(__shfl(v.re, src, 64), __shfl(v.im, src, 64)); }
__device__ inline cplx read_lane_c(cplx v, int lane) { return mk(read_lane(v.re, lane), read_lane(v.im, lane)); }

// A column norm as the pre-pivoting order takes it: one that is not a number counts as -1, behind
// every number. With the NaN itself no comparison would hold and columns would share a rank,
// which leaves entries of the permutation unset.
__device__ inline double order_norm(double v) { return v >= 0.0 ? v : -1.0; }

// Panel staging between A (global) and P (LDS, [NB][n], rows k0..n-1 of each column);
// logical column k is physical column perm[k] (perm == nullptr: the identity).
// Each thread moves one row of all NB columns per step: the NB loads are issued before
// any store, so memory latency is paid once per row rather than once per element.
// mode 0: P <- A as is; mode 1: P <- unit lower trapezoid (V with its implicit ones and
// zeros above the diagonal), columns t >= kb zero-filled.
template <int NB>
__device__ inline void stage_panel(cplx* P, const gcplx* A, const int* perm, int k0, int kb, int n, int tid,
                                   int mode, int cs = 0) {
  if (cs == 0) cs = n;  // LDS column stride of P
  const gcplx* src[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    const int k = k0 + min(t, kb - 1);
    src[t] = A + (size_t)(perm ? perm[k] : k) * n;
  }
  for (int r = k0 + tid; r < n; r += 256) {
    cplx v[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) v[t] = ld(src[t] + r);
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      cplx val = v[t];
      if (mode == 1) val = (t >= kb || r < k0 + t) ? mk(0, 0) : (r == k0 + t) ? mk(1, 0) : val;
      P[(size_t)t * cs + r] = val;
    }
  }
}

// ---------------------------------------------------------------------------
// k_qr_pipe<RQ>: the blocked QR with 8-column panels, RQ = ceil(nmax / 256) rows per thread.
//
// What bounds it is workgroup 0's chain of panels: apply panel p to panel p+1's columns, factor
// them, publish. The trailing updates run on the other workgroups and only have to keep up, so
// no barrier over the chain group is taken per panel. Instead
//   * block q (columns 8q .. 8q+7) belongs to workgroup 1 + q mod (W-1) for the whole
//     factorisation; its owner applies the panels to it in order;
//   * workgroup 0 publishes each panel (V in A, T in qr_Tf) by flags[0] = number of panels done;
//   * the owner of block p+2 publishes it after applying panel p (flags[1 + block]); workgroup
//     0 needs it one panel later and loads it while it writes panel p+1 back.
// With one group barrier per panel (all workgroups waiting for all) the loads, the barrier and
// the error-word read it took were about a third of a panel's time.
//
// A block is held as the C operand of v_mfma_f64_16x16x4: the 16 columns of a tile are the real
// (0-7) and imaginary (8-15) parts of the block's 8 columns, lane (li, lk) of wave w holds rows
// 16 (w + 4 tt) + 4 v + lk, column li. In that layout element v of a tile is also the B operand
// of k-step v of the same rows, so
//   [Vr Vi]^T [Xr Xi] (16 x 16, all four real products of V^H X at full tile use) and
//   X -= [Vr Vi] [[Zr Zi] [-Zi Zr]]
// take one MFMA per four rows each and no cross-lane sums; the vector form spent more time in
// its butterflies and lane broadcasts than in the products. For the column steps the panel moves
// through LDS (the buffer of V, free by then) to rows per thread, row off + tid + 256 q with
// off = n - 256 RQ: the first rows die first and finished rows are skipped.
//
// Measured (one chain, default workgroups, us per factorisation, one group barrier per panel and
// vector updates -> this): n = 64 163 -> 77, n = 256 631 -> 350, n = 400 1008 -> 730, n = 576
// 1850 -> 1320, n = 1024 5000 -> 3390. A panel at n = 400 takes 33,800 cycles: 15,700 in the eight
// column steps, 4,600 writing it back, 3,700 in V^H X, 3,300 for the next block's flag and loads,
// 2,100 each in the update, the move to rows and the wait for the loads. Above n = 512 a thread's
// rows and tiles exceed its 512 registers: RQ = 3 spills 18 (76 bytes per lane), RQ = 4 154 (548
// bytes), inside the panel chain; RQ = 1 and 2 spill none.
//
// WIDE: every trailing update of the launch is the 16-column one, workgroup 0's too when it is
// alone. It serves n > 512 with few workgroups per chain (launch_qr_blocked): one workgroup in the
// tile form waits for each block's loads in turn and was slower than the vector kernel that k_qr_pipe
// replaced (ms per factorisation, vector / tile form / this: n = 576 23.3 / 26.3 / 17.0, n = 1024 104 /
// 138 / 85), and with two to nine the instance without the block loop spills less (RQ = 4: 134
// registers; n = 1024, W = 2: 84 / 92 / 82, W = 4: 41 / 41 / 37; RQ = 3 the same either way).
// ---------------------------------------------------------------------------
// Bounded wait of a whole workgroup for *f >= want: thread 0 polls (relaxed loads, one acquire
// fence after the last), everyone learns the outcome through LDS. false: the wait timed out here
// or in another workgroup of the chain.
__device__ inline unsigned flag_load(const unsigned* f) {
  return __hip_atomic_load((const __attribute__((address_space(1))) unsigned*)f, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool wait_flag(const unsigned* f, unsigned want, int* error, int* s_fail) {
  if (threadIdx.x == 0) {
    int fail = 0;
    long long spins = 0;
    while (flag_load(f) < want) {
      if ((++spins & 31) == 0) {
        if (__hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
          fail = 1;
          break;
        }
        if (spins > kSpinLimit) {
          __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          fail = 1;
          break;
        }
      }
      __builtin_amdgcn_s_sleep(1);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    *s_fail = fail;
  }
  __syncthreads();
  return *s_fail == 0;
}
// this wave's outstanding global stores have completed (vmcnt(0), no wait for the LDS)
__device__ inline void wait_stores() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// one thread: publish *f = v after a barrier that every wave entered with its stores complete
// (write-through stores in place of the release fence cost more than the write-back: 8-byte
// agent-scope stores held workgroup 0 for 8,000 cycles a panel)
__device__ inline void set_flag(unsigned* f, unsigned v) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  __hip_atomic_store((__attribute__((address_space(1))) unsigned*)f, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// sqrt(s) and 1 / sqrt(s) of a normal s > 0: Goldschmidt's iteration from the hardware estimate,
// then one residual correction of each. One chain of ten dependent operations in place of a
// square root followed by a division.
__device__ inline void sqrt_rsqrt(double s, double& root, double& inv) {
  const double y = __builtin_amdgcn_rsq(s);
  double g = s * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  root = fma(fma(-g, g, s), h, g);
  const double i0 = h + h;
  inv = fma(i0, fma(-i0, root, 1.0), i0);
}
// 1 / x of a normal x: two Newton steps from the hardware estimate
__device__ inline double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  return fma(r, fma(-x, r, 1.0), r);
}

template <int RQ, bool WIDE>
__global__ __launch_bounds__(256) void k_qr_pipe(const ChainDesc* chains, MatRef Ar, VecRef Dr, int prepivot, int ps,
                                                 const int* bmap) {
  constexpr int NB = 8, V = 2 * NB, LS = 2;  // V doubles per butterfly; after it, lane l holds value l >> LS
  constexpr int TT = 4 * RQ;                 // 16-row tiles per wave
  // grid (W, chains), or with a block map a 1-D grid where block b serves chain bmap[b] & 0xFFFF
  // as workgroup (bmap[b] >> 16) & 0xFF of (bmap[b] >> 24) (workgroup counts per chain)
  const int bm = bmap ? bmap[blockIdx.x] : 0;
  const ChainDesc& c = chains[bmap ? (bm & 0xFFFF) : blockIdx.y];
  const int n = c.n;
  const int W = bmap ? (bm >> 24) & 0xFF : gridDim.x, w = bmap ? (bm >> 16) & 0xFF : blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = 4;
  const int li = lane & 15, lk = lane >> 4, lu = li & 7, lim = li >> 3;
  gcplx* A = gp(matptr(c, Ar));
  gdouble* D = gp(vecptr(c, Dr));
  // (every pointer of the descriptor once: a store could change it for all the compiler knows, and
  // each re-read waits for every load and store in flight)
  gcplx *Tf = gp(c.qr_Tf), *taug = gp(c.qr_tau);
  unsigned* flags = c.qr_flags;
  int* err = c.error;
  const GroupSync g{c.bar_count, c.bar_gen, c.error, (unsigned int)W};
  const int nblk = (n + NB - 1) / NB;
  const int off = n - 256 * RQ;
  // with many columns per trailing workgroup (at least 128 at the start) a wave takes 16 of them
  // at a time instead of the workgroup 8: no barriers, but X streams from memory twice (WIDE: always)
  const bool mt = WIDE || (W > 1 && n >= 128 * (W - 1));

  extern __shared__ double smem[];
  cplx* P = reinterpret_cast<cplx*>(smem);  // [NB][ps] panel V (rows k0..n-1 used, row r at 16 + r)
  // [2][4][2][64] per-wave partial W of the tile form (two halves by turns, see apply_tiles);
  // [4][8][16] W of the 16-column trailing update
  double* part = reinterpret_cast<double*>(P + (size_t)NB * ps);
  cplx* wscr = reinterpret_cast<cplx*>(part);
  __shared__ int perm[kQrMaxN], lpos[kQrMaxN];
  __shared__ cplx Tl[NB * NB];     // Tl[j * NB + t] = T(j, t) of the panel in P
  __shared__ cplx rowb[NB * NB];   // rows k0 .. k0+7 of the panel being factored: R and V
  __shared__ double4 red[2][V];    // sums of a panel step, by step parity: one partial per wave
  __shared__ cplx piv[2][NB];      // the pivot row of a panel step, by step parity
  __shared__ int s_fail;

  // ---- the flags of this factorisation, visible to all before the first wait
  if (w == 0)
    for (int e = tid; e <= nblk; e += 256) __hip_atomic_store(flags + e, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // ---- column order
  if (prepivot) {
    for (int col = w + W * wave; col < n; col += W * nwaves) {
      const gcplx* a = A + (size_t)col * n;
      double acc = 0.0;
      for (int k = lane; k < n; k += 64) acc += abs2(ld(a + k));
      acc = wave_sum(acc);
      if (lane == 0) gp(c.qr_vn)[col] = sqrt(acc);
    }
  }
  wait_stores();
  group_sync(g);
  if (group_failed(g)) return;
  if (prepivot) {
    double* vn = reinterpret_cast<double*>(P);  // n doubles, before the panel buffer is used
    for (int k = tid; k < n; k += blockDim.x) vn[k] = order_norm(gp(c.qr_vn)[k]);
    __syncthreads();
    for (int col = tid; col < n; col += blockDim.x) {
      const double v = vn[col];
      int r = 0;
      for (int q = 0; q < n; ++q) {
        const double u = vn[q];
        r += (u > v || (u == v && q < col)) ? 1 : 0;
      }
      lpos[col] = r;
    }
    __syncthreads();
    for (int col = tid; col < n; col += blockDim.x) perm[lpos[col]] = col;
  } else {
    for (int k = tid; k < n; k += blockDim.x) perm[k] = lpos[k] = k;
  }
  __syncthreads();

  // Every V in P starts at LDS row 16 + k0 with 16 zero rows before it, so that the tile which
  // straddles row k0 (tiles end at row n - 1, not at multiples of 16 from row 0) needs no masks:
  // its rows before k0 meet zeros, and keep the finite values they have.
  v4d X[TT];        // a block in tile layout
  cplx x[RQ][NB];   // the panel being factored, rows per thread
  // this thread's rows, re-read per panel: as loop invariants the unrolled addresses and masks
  // below would be formed once and spill
  int tr = off + 16 * wave + lk, ta = off + 16 * wave + li, tx = off + tid;
  // first tile of this wave that reaches row k
  auto first_tile = [&](int k) __attribute__((always_inline)) { return ((max(k - off, 0) >> 4) - wave + 3) >> 2; };

  // the tiles of the block at logical column kc that reach row kr into X (columns past the last
  // one repeat it: nothing reads them)
  auto load_tiles = [&](int kc, int kr) __attribute__((always_inline)) {
    const int kbc = min(NB, n - kc), t0 = first_tile(kr);
    const gdouble* a = (const gdouble*)(A + (size_t)perm[kc + min(lu, kbc - 1)] * n) + lim;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt >= t0) {
#pragma unroll
        for (int v = 0; v < 4; ++v) X[tt][v] = a[2 * max(tr + 64 * tt + 4 * v, 0)];
      } else {
        X[tt] = v4d{0.0, 0.0, 0.0, 0.0};  // (defined on every path: not live during the column steps)
      }
  };
  auto store_tiles = [&](int kc, int kr) __attribute__((always_inline)) {
    const int t0 = first_tile(kr);
    gdouble* a = (gdouble*)(A + (size_t)perm[min(kc + lu, n - 1)] * n) + lim;
    const int lo = lu < n - kc ? kr : n;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt >= t0) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (tr + 64 * tt + 4 * v >= lo) a[2 * (tr + 64 * tt + 4 * v)] = X[tt][v];
      }
  };
  // X <- (I - V T^H V^H) X with V (rows >= k0) in P and T in Tl. Nothing but the barrier in here
  // orders one block against the next, so a wave that is ahead writes the next block's partial
  // sums while another still reads this block's: they alternate between two halves of `part`, and
  // a half is written again only behind the barrier of the block between.
  int half = 0;
  auto apply_tiles = [&](int k0) __attribute__((always_inline)) {
    const int t0 = first_tile(k0);
    v4d acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
    const double* pv = reinterpret_cast<const double*>(P + (size_t)lu * ps + 16 + tr) + lim;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt >= t0) {
        acc0 = mfma4(pv[2 * (64 * tt)], X[tt][0], acc0);
        acc1 = mfma4(pv[2 * (64 * tt + 4)], X[tt][1], acc1);
        acc0 = mfma4(pv[2 * (64 * tt + 8)], X[tt][2], acc0);
        acc1 = mfma4(pv[2 * (64 * tt + 12)], X[tt][3], acc1);
      }
    // Lane (li, lk): row l = lk (lk + 4 for w1) of W = V^H X, component li, from the products
    // Vr Xr + Vi Xi (li < 8) and Vr Xi - Vi Xr (li >= 8); Vi's rows are 8 further down the tile,
    // the other component is 8 lanes away. Then the sum over the waves.
    const double o0 = dpp_move<0x128>(acc0[2] + acc1[2]), o1 = dpp_move<0x128>(acc0[3] + acc1[3]);  // row_ror:8
    double* sums = part + half;
    half ^= 512;
    sums[wave * 128 + lane] = (acc0[0] + acc1[0]) + (lim ? -o0 : o0);
    sums[wave * 128 + 64 + lane] = (acc0[1] + acc1[1]) + (lim ? -o1 : o1);
    __syncthreads();
    const double w0 = (sums[lane] + sums[128 + lane]) + (sums[256 + lane] + sums[384 + lane]);
    const double w1 = (sums[64 + lane] + sums[192 + lane]) + (sums[320 + lane] + sums[448 + lane]);
    // That is the B operand of Z = T^H W: [Zr Zi] = Tr^T [Wr Wi] + Ti^T [Wi -Wr], and element 0
    // (1) of the product is row lk (lk + 4) of [Zr Zi], the B operand of the update
    const cplx t0l = Tl[lk * NB + lu], t1l = Tl[(lk + 4) * NB + lu];
    const double x0 = dpp_move<0x128>(w0), x1 = dpp_move<0x128>(w1);
    v4d z = {0.0, 0.0, 0.0, 0.0};
    z = mfma4(lim ? 0.0 : t0l.re, w0, z);
    z = mfma4(lim ? 0.0 : t1l.re, w1, z);
    z = mfma4(lim ? 0.0 : t0l.im, lim ? -x0 : x0, z);
    z = mfma4(lim ? 0.0 : t1l.im, lim ? -x1 : x1, z);
    // rows of [[Zr Zi] [-Zi Zr]], negated: k-steps 0, 1 (Vr) and 2, 3 (Vi)
    const double y0 = dpp_move<0x128>(z[0]), y1 = dpp_move<0x128>(z[1]);
    const double b0 = -z[0], b1 = -z[1], b2 = lim ? -y0 : y0, b3 = lim ? -y1 : y1;
    const cplx* pa = P + (size_t)lk * ps + 16 + ta;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt >= t0) {
        const cplx v0 = pa[64 * tt], v1 = pa[(size_t)4 * ps + 64 * tt];
        X[tt] = mfma4(v0.re, b0, X[tt]);
        X[tt] = mfma4(v1.re, b1, X[tt]);
        X[tt] = mfma4(v0.im, b2, X[tt]);
        X[tt] = mfma4(v1.im, b3, X[tt]);
      }
  };
  // the published panel at k0 into P as the unit lower trapezoid V, every load before any store
  auto stage_V = [&](int k0) __attribute__((always_inline)) {
    const int q0 = max(k0 - off, 0) >> 8;
    cplx y[RQ][NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const gcplx* a = A + (size_t)perm[k0 + t] * n;
#pragma unroll
      for (int q = 0; q < RQ; ++q)
        if (q >= q0) {
          const gcplx* src = a + max(tx + 256 * q, k0);
          y[q][t].re = src->re;
          y[q][t].im = src->im;
        }
    }
#pragma unroll
    for (int q = 0; q < RQ; ++q)
      if (q >= q0) {
        const int r = tx + 256 * q;
        if (r >= k0) {
#pragma unroll
          for (int t = 0; t < NB; ++t) {
            P[(size_t)t * ps + 16 + r].re = r < k0 + t ? 0.0 : r == k0 + t ? 1.0 : y[q][t].re;
            P[(size_t)t * ps + 16 + r].im = r <= k0 + t ? 0.0 : y[q][t].im;
          }
        }
      }
    if (tid >= 128) P[(size_t)((tid - 128) >> 4) * ps + k0 + (tid & 15)] = mk(0, 0);  // rows k0 - 16 .. k0 - 1
  };
  // the panel at k1, tiles of X that reach row kr, through P into x: rows >= k1 to x (zero before
  // that; LDS row 0 is zero throughout), rows kr .. k1 - 1 of R to A
  auto tiles_to_rows = [&](int k1, int kr) __attribute__((always_inline)) {
    const int t0 = first_tile(kr);
    double* pd = reinterpret_cast<double*>(P + (size_t)lu * ps + 16 + tr) + lim;
    __syncthreads();  // every wave has read V
#pragma unroll
    for (int tt = 0; tt < TT; ++tt)
      if (tt >= t0) {
#pragma unroll
        for (int v = 0; v < 4; ++v) pd[2 * (64 * tt + 4 * v)] = X[tt][v];
      }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const int r = tx + 256 * q;
      const cplx* src = P + (r >= k1 ? 16 + r : 0);
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        x[q][t].re = src[(size_t)t * ps].re;
        x[q][t].im = src[(size_t)t * ps].im;
      }
    }
    const int t = tid >> 3, r = kr + (tid & 7);
    if (tid < NB * NB && r < k1 && k1 + t < n) {
      const cplx* src = P + (size_t)t * ps + 16 + r;
      st(A + (size_t)perm[k1 + t] * n + r, mk(src->re, src->im));
    }
  };
  // ---- the column steps of the panel at logical column k0, held in x. Per column t (zlarfg,
  // then H^H on the columns after it):
  //   the owner of the pivot row i = k0 + t moves it to LDS and clears its columns >= t, so rows
  //   above the diagonal need no masks;
  //   one butterfly sums |x_t|^2 and x_t^H a_u (u > t) over the rows below the pivot, plus
  //   v_j^H x_t (j < t) for zlarft; after one barrier every thread forms beta, tau and
  //   1 / (alpha - beta) from the same sums and updates its rows; wave 0 keeps row i of R and V;
  //   column t of T (zlarft, forward and columnwise): S(j, t) = v_j^H v_t = conj(v_j(i)) +
  //   v_j^H x_t / (alpha - beta), T(t, t) = tau, T(0:t, t) = -tau T(0:t, 0:t) S(0:t, t), lane j of
  //   every 16 keeping row j, so that T is ready with the last column.
  // A step is one wave per SIMD working through a chain of dependent operations, about 200
  // instructions: its length is what counts, so sums, pivot entries and factors stay one per lane
  // until the broadcasts, the square root also gives 1 / beta, and the factors of the update
  // need no other division.
  cplx trow[NB];   // lane j (of 16): row j of T
  auto column_steps = [&](int k0) __attribute__((always_inline)) {
    const int q0 = max(k0 - off, 0) >> 8;  // rows of x[q], q < q0, are finished
    const int kl = lane & 15;
    static_for<0, NB>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value, par = t & 1;
      const int i = k0 + t;
      double v[V];
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = 0.0;
#pragma unroll
      for (int q = 0; q < RQ; ++q)
        if (q >= q0) {
          if (tx + 256 * q == i) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
              piv[par][u].re = x[q][u].re;
              piv[par][u].im = x[q][u].im;
            }
#pragma unroll
            for (int u = t; u < NB; ++u) x[q][u] = mk(0, 0);
          }
          const cplx xt = x[q][t];
          v[0] = fma(xt.re, xt.re, fma(xt.im, xt.im, v[0]));
#pragma unroll
          for (int u = t + 1; u < NB; ++u) {
            const int e = 1 + 2 * (u - t - 1);
            v[e] = fma(xt.re, x[q][u].re, fma(xt.im, x[q][u].im, v[e]));
            v[e + 1] = fma(xt.re, x[q][u].im, fma(-xt.im, x[q][u].re, v[e + 1]));
          }
#pragma unroll
          for (int j = 0; j < t; ++j) {  // v_j^H x_t below the pivot, for S(j, t)
            const int e = 1 + 2 * (NB - 1 - t) + 2 * j;
            v[e] = fma(x[q][j].re, xt.re, fma(x[q][j].im, xt.im, v[e]));
            v[e + 1] = fma(x[q][j].re, xt.im, fma(-x[q][j].im, xt.re, v[e + 1]));
          }
        }
      wave_reduce_scatter<V>(v);
      if ((lane & ((1 << LS) - 1)) == 0) reinterpret_cast<double*>(&red[par][lane >> LS])[wave] = v[0];
      __syncthreads();
      // lane k of every row of 16: its complex sum, of column t+1+k (k < NB-1-t) or of reflector
      // k - (NB-1-t), and that column's entry of the pivot row
      const int k = min(kl, NB - 2), m = k < NB - 1 - t ? t + 1 + k : k - (NB - 1 - t);
      const double4 q0s = red[par][0], qr = red[par][1 + 2 * k], qi = red[par][2 + 2 * k];
      const cplx alpha = mk(piv[par][t].re, piv[par][t].im), pm = mk(piv[par][m].re, piv[par][m].im);
      const double xsq = (q0s.x + q0s.y) + (q0s.z + q0s.w);
      const cplx raw = mk((qr.x + qr.y) + (qr.z + qr.w), (qi.x + qi.y) + (qi.z + qi.w));
      // zlarfg: H^H (alpha, x) = (beta, 0), v = (1, x / d), d = alpha - beta, tau = -d / beta.
      // With nothing below the pivot and a real alpha H = I: 1 / beta is taken as 0, which makes
      // tau and f zero, and x is zero whatever d is.
      const bool none = xsq == 0.0 && alpha.im == 0.0;
      const double ssq = fma(alpha.re, alpha.re, fma(alpha.im, alpha.im, xsq));
      double nrm, inv;
      sqrt_rsqrt(none ? 1.0 : ssq, nrm, inv);
      const double ib = none ? 0.0 : -copysign(inv, alpha.re);
      const double beta = none ? alpha.re : -copysign(nrm, alpha.re);
      const cplx d = mk(alpha.re + copysign(nrm, alpha.re), alpha.im);
      // v^H a_u = a_u(i) + conj(1 / d) x_t^H a_u, times conj(tau) = -conj(d) / beta:
      // f = -(conj(d) a_u(i) + x_t^H a_u) / beta, which needs no division by |d|^2
      cplx fl = raw;
      cfma_cj(fl, d, pm);
      fl = mk(-ib * fl.re, -ib * fl.im);
      const double id = recip(fma(d.re, d.re, d.im * d.im));  // |d|^2 <= 4 (|alpha|^2 + xsq)
      const cplx sc = mk(d.re * id, -d.im * id), tau = mk(-d.re * ib, -d.im * ib);
      cplx f[NB];
      static_for<t + 1, NB>([&](auto uc) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        f[u] = mk(dpp_move<0x150 + (u - t - 1)>(fl.re), dpp_move<0x150 + (u - t - 1)>(fl.im));  // row_newbcast
      });
#pragma unroll
      for (int q = 0; q < RQ; ++q)
        if (q >= q0) {
          const cplx vt = sc * x[q][t];
#pragma unroll
          for (int u = t + 1; u < NB; ++u) {
            x[q][u].re = fma(-f[u].re, vt.re, fma(f[u].im, vt.im, x[q][u].re));
            x[q][u].im = fma(-f[u].re, vt.im, fma(-f[u].im, vt.re, x[q][u].im));
          }
          x[q][t] = vt;
        }
      if (tid < NB) {  // row i of R (columns >= t) and of V (columns < t)
        const bool diag = tid == NB - 1, r = k < NB - 1 - t;
        rowb[t * NB + (diag ? t : m)].re = diag ? beta : r ? pm.re - fl.re : pm.re;
        rowb[t * NB + (diag ? t : m)].im = diag ? 0.0 : r ? pm.im - fl.im : pm.im;
      }
      cplx sj = conj(pm), acc = mk(0, 0);
      cfma(sj, sc, raw);
      static_for<0, t>([&](auto lc) __attribute__((always_inline)) {
        constexpr int l = decltype(lc)::value, src = NB - 1 - t + l;
        cfma(acc, trow[l], mk(dpp_move<0x150 + src>(sj.re), dpp_move<0x150 + src>(sj.im)));
      });
      acc = -(tau * acc);  // (zero on the lanes j >= t)
      trow[t].re = kl == t ? tau.re : acc.re;
      trow[t].im = kl == t ? tau.im : acc.im;
    });
  };
  // ---- the factored panel p at k0: V to P, T to Tl; rows >= k0 to A, tau, D and T to global memory
  auto write_panel = [&](int k0, int p) __attribute__((always_inline)) {
    const int kb = min(NB, n - k0);
    gcplx* Tg = Tf + (size_t)p * NB * NB;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      gcplx* a = A + (size_t)perm[k0 + min(t, kb - 1)] * n;
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = tx + 256 * q;
        const cplx xv = x[q][t];
        if (r >= k0 + NB) {
          P[(size_t)t * ps + 16 + r].re = xv.re;
          P[(size_t)t * ps + 16 + r].im = xv.im;
        }
        if (t < kb && r >= k0 + NB) st(a + r, xv);
      }
    }
    if (wave == 3) {  // lane (t, u): rows k0 .. k0+7
      const int t = lane >> 3, u = lane & 7;
      const cplx e = mk(rowb[lane].re, rowb[lane].im);
      if (k0 + t < n) {
        P[(size_t)u * ps + 16 + k0 + t].re = u < t ? e.re : u == t ? 1.0 : 0.0;
        P[(size_t)u * ps + 16 + k0 + t].im = u < t ? e.im : 0.0;
        if (u < kb) st(A + (size_t)perm[k0 + u] * n + k0 + t, e);
        if (t == u) D[k0 + t] = fabs(e.re);
      }
    }
    if (tid >= 64 && tid < 192) P[(size_t)((tid - 64) >> 4) * ps + k0 + (tid & 15)] = mk(0, 0);  // rows k0 - 16 .. k0 - 1
    if (tid < NB) {  // row tid of T
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        const bool ok = t < kb && tid < kb;
        const cplx v = mk(ok ? trow[t].re : 0.0, ok ? trow[t].im : 0.0);
        Tl[tid * NB + t].re = v.re;
        Tl[tid * NB + t].im = v.im;
        st(Tg + tid * NB + t, v);
      }
    }
    if (tid < kb) {  // tau: T's diagonal
      const cplx v = mk(Tl[tid * (NB + 1)].re, Tl[tid * (NB + 1)].im);
      st(taug + k0 + tid, v);
    }
  };
  const int ws = W == 1 ? 1 : W - 1;  // workgroups of the trailing blocks
  // Trailing update of panel p (rows >= k0) on the matrix cores (mt), for workgroups w >= 1 or the
  // only one: the own blocks from fb on in tiles of two blocks, 16 columns, tile q to wave q mod 4.
  // Per tile: W = V^H X (K = rows, A(i, k) = conj V(r, i), B(k, j) = X(r, col_j)), then
  // Z = T^H W with the vector units (lane (j, k) forms Z(k, j) and Z(k + 4, j), exactly its B
  // operands of the second product), then X -= V Z in 16-row tiles. X streams from global
  // memory twice (loads four steps ahead); V comes from P (stride ps: conflict-free). When fb is
  // the block workgroup 0 waits for, wave 0 publishes it after the tile that holds it.
  auto trailing_mfma = [&](int k0, int fb, int need) __attribute__((always_inline)) {
    const int vi = min(li, NB - 1);
    const int nbw = fb < nblk ? (nblk - 1 - fb) / ws + 1 : 0;
    const int nst = (n - k0) >> 2;
    cplx* wsc = wscr + wave * 128;
    for (int q = wave; 2 * q < nbw; q += nwaves) {
      const int j = 2 * q + (li >> 3);
      const int cl = (fb + j * ws) * NB + (li & 7);
      const bool valid = j < nbw && cl < n;
      gcplx* a = A + (size_t)perm[valid ? cl : n - 1] * n;
      v4d wr = {0.0, 0.0, 0.0, 0.0}, wi = {0.0, 0.0, 0.0, 0.0};
      constexpr int PF = 8;  // k-steps of X loaded ahead of the products
      cplx xb[PF];
#pragma unroll
      for (int u = 0; u < PF; ++u) xb[u] = ld(a + k0 + 4 * min(u, nst - 1) + lk);
      for (int s0 = 0; s0 < nst; s0 += PF) {
        cplx xc[PF];
#pragma unroll
        for (int u = 0; u < PF; ++u) xc[u] = xb[u];
#pragma unroll
        for (int u = 0; u < PF; ++u) xb[u] = ld(a + k0 + 4 * min(s0 + PF + u, nst - 1) + lk);
#pragma unroll
        for (int u = 0; u < PF; ++u) {
          if (s0 + u < nst) {
            const cplx v = P[(size_t)vi * ps + 16 + k0 + 4 * (s0 + u) + lk];
            const double vr = li < NB ? v.re : 0.0, vm = li < NB ? v.im : 0.0;
            const double xr = valid ? xc[u].re : 0.0, xm = valid ? xc[u].im : 0.0;
            // W += V^H X: re += Vr Xr + Vi Xi, im += Vr Xi - Vi Xr
            wr = mfma4(vr, xr, wr);
            wi = mfma4(vr, xm, wi);
            wr = mfma4(vm, xm, wr);
            wi = mfma4(-vm, xr, wi);
          }
        }
      }
      // lane (li, lk) holds W(lk, li) and W(lk + 4, li); every lane needs W(:, li)
      wsc[lk * 16 + li] = mk(wr[0], wi[0]);
      wsc[(lk + 4) * 16 + li] = mk(wr[1], wi[1]);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      cplx z0 = mk(0, 0), z1 = mk(0, 0);
#pragma unroll
      for (int l = 0; l < NB; ++l) {
        const cplx wl = wsc[l * 16 + li];
        cfma_cj(z0, Tl[l * NB + lk], wl);
        cfma_cj(z1, Tl[l * NB + lk + 4], wl);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // W read before the next tile writes it
      // X -= V Z over 16-row tiles: element v of lane (li, lk) is row r0 + lk + 4 v, column li
      cplx cb[4], cn[4];  // the next two row tiles' X, loaded ahead
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        cb[v] = ld(a + min(k0 + lk + 4 * v, n - 1));
        cn[v] = ld(a + min(k0 + 16 + lk + 4 * v, n - 1));
      }
      for (int r0 = k0; r0 < n; r0 += 16) {
        v4d dr, di;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          dr[v] = cb[v].re;
          di[v] = cb[v].im;
          cb[v] = cn[v];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) cn[v] = ld(a + min(r0 + 32 + lk + 4 * v, n - 1));
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const int ra = r0 + li;
          const cplx a0 = P[(size_t)(4 * ks + lk) * ps + 16 + min(ra, n - 1)];
          const double ar = ra < n ? a0.re : 0.0, am = ra < n ? a0.im : 0.0;
          const cplx z = ks ? z1 : z0;
          // X -= V Z: re += -Vr Zr + Vi Zi, im += -Vr Zi - Vi Zr
          dr = mfma4(-ar, z.re, dr);
          di = mfma4(-ar, z.im, di);
          dr = mfma4(am, z.im, dr);
          di = mfma4(-am, z.re, di);
        }
        if (valid) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int row = r0 + lk + 4 * v;
            if (row < n) {
              st(a + row, mk(dr[v], di[v]));
            }
          }
        }
      }
      if (q == 0 && fb == need) {  // (tile 0 is wave 0's: the wave publishes its own stores)
        wait_stores();
        if (lane == 0) set_flag(flags + 1 + need, 1u);
      }
    }
  };

  // the rows before row 0: a panel's rows per thread reach them, and they have to be finite
  if (tid < 128) P[(size_t)(tid >> 4) * ps + (tid & 15)] = mk(0, 0);
  int own = w - 1;
  bool loaded = false;  // the next block's tiles are already in X
  for (int p = -1, k1 = 0; k1 < n; ++p, k1 += NB) {  // apply panel p, factor panel p+1 at k1
    const int k0 = max(k1 - NB, 0);
    asm volatile("" : "+v"(tr), "+v"(ta), "+v"(tx));
    // the first own block beyond panel p+1 (workgroup 0 owns none unless it is alone)
    int fb = nblk;
    if (W > 1 && w != 0) loaded = true;
    if (W == 1) {
      fb = p < 0 ? nblk : p + 2;
      if (WIDE && fb < nblk) {
        trailing_mfma(k0, fb, -1);
        __syncthreads();  // wscr is in part's place
        fb = nblk;
      }
    } else if (w != 0) {
      if (p < 0) continue;
      while (own < p + 2) own += ws;
      fb = own;
      if (fb >= nblk) return;  // no block of this workgroup is left
      if (!mt) load_tiles(fb * NB, k0);  // (own columns: before the panel is there)
      if (!wait_flag(flags, (unsigned)(p + 1), err, &s_fail)) return;
      stage_V(k0);
      if (tid < NB * NB) Tl[tid] = ld(Tf + (size_t)p * NB * NB + tid);
      __syncthreads();
      if (mt) {
        trailing_mfma(k0, fb, p + 2);
        continue;
      }
    }
    // the own trailing blocks first, then, on workgroup 0, panel p+1 itself, which stays in X
    // (WIDE: the panel alone)
    if (WIDE) fb = nblk;
    for (;; fb += ws) {
      const bool next = fb >= nblk;
      if (next && w != 0) break;
      const int kc = next ? k1 : fb * NB;
      if (!loaded) load_tiles(kc, k0);
      if (p >= 0) apply_tiles(k0);
      if (next) break;
      store_tiles(kc, k0);
      if (W > 1 && fb == p + 2) {
        wait_stores();
        __syncthreads();
        if (tid == 0) set_flag(flags + 1 + fb, 1u);
      }
      loaded = false;
    }
    if (w != 0) continue;
    tiles_to_rows(k1, k0);
    const bool fetch = W > 1 && k1 + NB < n, need = fetch && p >= 0;
    column_steps(k1);
    if (need) {
      // block p+2 carries panel p; its owner has had a panel's time to bring it up to date
      if (!wait_flag(flags + 1 + (p + 2), 1u, err, &s_fail)) return;
    } else {
      __syncthreads();
    }
    if (fetch) load_tiles(k1 + NB, k1);
    loaded = fetch;
    write_panel(k1, p + 1);
    wait_stores();
    __syncthreads();
    if (W > 1 && tid == 192) set_flag(flags, (unsigned)(p + 2));
  }
  if (w == 0) {
    for (int k = tid; k < n; k += blockDim.x) {
      gp(c.qr_perm)[k] = perm[k];
      gp(c.qr_lpos)[k] = lpos[k];
    }
  }
}

// k_qr_blocked<NB, RQ>: the same factorisation by one group barrier per panel, on the vector
// units; it serves 16-column panels (twice the panel does not fit k_qr_pipe's tiles).
// Workgroup 0's panel work keeps the panel in registers: thread tid owns rows r = tid + 256 q
// (q < RQ) of the NB panel columns. Every cross-thread sum goes through one butterfly
// reduce-scatter per wave and one LDS exchange, so a panel column costs one barrier.
// Selections below are written without data-dependent branches around loads: a guard
// around each LDS read makes the compiler wait for it before the next one.
template <int NB, int RQ>
__global__ __launch_bounds__(256) void k_qr_blocked(const ChainDesc* chains, MatRef Ar, VecRef Dr, int prepivot,
                                                    int ps, const int* bmap) {
  constexpr int V = 2 * NB;               // doubles per butterfly
  constexpr int LS = 1;                   // after it, lane l holds value l >> LS
  static_assert(NB == 16, "");
  // grid (W, chains), or with a block map a 1-D grid where block b serves chain bmap[b] & 0xFFFF
  // as workgroup (bmap[b] >> 16) & 0xFF of (bmap[b] >> 24) (workgroup counts per chain)
  const int bm = bmap ? bmap[blockIdx.x] : 0;
  const ChainDesc& c = chains[bmap ? (bm & 0xFFFF) : blockIdx.y];
  const int n = c.n;
  const int W = bmap ? (bm >> 24) & 0xFF : gridDim.x, w = bmap ? (bm >> 16) & 0xFF : blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nwaves = blockDim.x >> 6;
  gcplx* A = gp(matptr(c, Ar));
  gdouble* D = gp(vecptr(c, Dr));
  const GroupSync g{c.bar_count, c.bar_gen, c.error, (unsigned int)W};

  extern __shared__ double smem[];
  cplx* P = reinterpret_cast<cplx*>(smem);  // [NB][ps] panel V (rows k0..n-1 used)
  __shared__ int perm[kQrMaxN], lpos[kQrMaxN];
  __shared__ cplx Tl[NB * NB];  // Tl[j * NB + t] = T(j, t)
  __shared__ cplx taul[NB];
  __shared__ double betal[NB];
  __shared__ double red[2][4][V];     // per-wave sums of a panel step, by step parity
  __shared__ cplx piv[2][NB];         // the pivot row of a panel step, by step parity
  __shared__ double redW[4][NB][V + 1];  // per-wave V^H a of NB columns (padded: no bank conflicts)

  // ---- column order
  if (prepivot) {
    for (int col = w + W * wave; col < n; col += W * nwaves) {
      const gcplx* a = A + (size_t)col * n;
      double acc = 0.0;
      for (int k = lane; k < n; k += 64) acc += abs2(ld(a + k));
      acc = wave_sum(acc);
      if (lane == 0) gp(c.qr_vn)[col] = sqrt(acc);
    }
    group_sync(g);
    if (group_failed(g)) return;
    double* vn = reinterpret_cast<double*>(P);  // n doubles, before the panel buffer is used
    for (int k = tid; k < n; k += blockDim.x) vn[k] = order_norm(gp(c.qr_vn)[k]);
    __syncthreads();
    for (int col = tid; col < n; col += blockDim.x) {
      const double v = vn[col];
      int r = 0;
      for (int q = 0; q < n; ++q) {
        const double u = vn[q];
        r += (u > v || (u == v && q < col)) ? 1 : 0;
      }
      lpos[col] = r;
    }
    __syncthreads();
    for (int col = tid; col < n; col += blockDim.x) perm[lpos[col]] = col;
  } else {
    for (int k = tid; k < n; k += blockDim.x) perm[k] = lpos[k] = k;
  }
  __syncthreads();

  cplx x[RQ][NB];  // this thread's rows of the panel being factored

  // rows >= kr of logical columns kc .. kc+kbc-1 into x (everything else zero)
  auto load_regs = [&](int kc, int kbc, int kr) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const gcplx* a = A + (size_t)perm[kc + min(t, kbc - 1)] * n;
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = tid + 256 * q;
        const gcplx* src = a + min(r, n - 1);
        const cplx v = mk(src->re, src->im);
        x[q][t] = (t < kbc && r >= kr && r < n) ? v : mk(0, 0);
      }
    }
  };

  // ---- factor the panel at logical column k0 (panel index p) held in x; rows >= kw of x are
  // valid and written back. Per column t (zlarfg, then H^H on the columns after it):
  //   one butterfly sums |x_t|^2 and x_t^H a_u (u > t) over the rows below the pivot, plus
  //   v_j^H x_t (j < t) for zlarft; the pivot row goes through LDS; after one barrier every
  //   thread forms beta, tau and 1/(alpha - beta) from the same sums and updates its rows:
  //   v^H a_u = a_u(i) + conj(1/(alpha - beta)) x_t^H a_u, and wave 0 stores
  //   S(j, t) = v_j^H v_t = conj(v_j(i)) + (1/(alpha - beta)) v_j^H x_t.
  // Every call site of this and of the block update below is single, and the kernel's code
  // fits the instruction cache: the panel loop runs without instruction fetch stalls.
  auto factor_regs = [&](int k0, int p, int kw) __attribute__((always_inline)) {
    const int kb = min(NB, n - k0);
    gcplx* Tg = gp(c.qr_Tf) + (size_t)p * NB * NB;
    static_for<0, NB>([&](auto tc) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value, par = t & 1;
      const int i = k0 + t;
      double v[V];
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = 0.0;
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = tid + 256 * q;
        const cplx xt = (r > i) ? x[q][t] : mk(0, 0);
        v[0] += abs2(xt);
#pragma unroll
        for (int u = t + 1; u < NB; ++u) {
          const int e = 1 + 2 * (u - t - 1);
          v[e] = fma(xt.re, x[q][u].re, fma(xt.im, x[q][u].im, v[e]));
          v[e + 1] = fma(xt.re, x[q][u].im, fma(-xt.im, x[q][u].re, v[e + 1]));
        }
#pragma unroll
        for (int j = 0; j < t; ++j) {  // v_j^H x_t below the pivot, for S(j, t)
          const int e = 1 + 2 * (NB - 1 - t) + 2 * j;
          v[e] = fma(x[q][j].re, xt.re, fma(x[q][j].im, xt.im, v[e]));
          v[e + 1] = fma(x[q][j].re, xt.im, fma(-x[q][j].im, xt.re, v[e + 1]));
        }
      }
#pragma unroll
      for (int q = 0; q < RQ; ++q)
        if (tid + 256 * q == i) {  // the owner of the pivot row (all columns: v_j(i) for j < t too)
#pragma unroll
          for (int u = 0; u < NB; ++u) {
            piv[par][u].re = x[q][u].re;
            piv[par][u].im = x[q][u].im;
          }
        }
      wave_reduce_scatter<V>(v);
      if ((lane & ((1 << LS) - 1)) == 0) red[par][wave][lane >> LS] = v[0];
      __syncthreads();
      const double xsq = (red[par][0][0] + red[par][1][0]) + (red[par][2][0] + red[par][3][0]);
      const cplx alpha = mk(piv[par][t].re, piv[par][t].im);
      cplx tau, sc;
      double beta;
      // zlarfg: H^H (alpha, x) = (beta, 0), v = (1, x / (alpha - beta))
      if (xsq == 0.0 && alpha.im == 0.0) {
        tau = mk(0, 0);
        beta = alpha.re;
        sc = mk(1, 0);
      } else {
        beta = -copysign(sqrt(alpha.re * alpha.re + alpha.im * alpha.im + xsq), alpha.re);
        const double ib = 1.0 / beta;  // two divisions on the per-column critical path, not five
        tau = mk((beta - alpha.re) * ib, -alpha.im * ib);
        const cplx d = alpha - mk(beta, 0);  // |d|^2 <= 4 (|alpha|^2 + xsq): no new overflow
        const double id = 1.0 / (d.re * d.re + d.im * d.im);
        sc = mk(d.re * id, -d.im * id);
      }
      // lane k forms f for column t+1+k (its sums read by lane), then every lane takes them
      // from scalar registers
      cplx fl;
      {
        const int k = min(lane, NB - 1 - t > 0 ? NB - 2 - t : 0), e = 1 + 2 * k;
        const cplx raw = mk((red[par][0][e] + red[par][1][e]) + (red[par][2][e] + red[par][3][e]),
                            (red[par][0][e + 1] + red[par][1][e + 1]) + (red[par][2][e + 1] + red[par][3][e + 1]));
        const int u = min(t + 1 + k, NB - 1);
        cplx dot = mk(piv[par][u].re, piv[par][u].im);
        cfma_cj(dot, sc, raw);
        fl = conj(tau) * dot;
      }
      cplx f[NB];
#pragma unroll
      for (int u = t + 1; u < NB; ++u) f[u] = read_lane_c(fl, u - t - 1);
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = tid + 256 * q;
        const cplx xt = x[q][t];
        const cplx vt = (r > i) ? sc * xt : (r == i) ? mk(1, 0) : mk(0, 0);
#pragma unroll
        for (int u = t + 1; u < NB; ++u) x[q][u] = x[q][u] - f[u] * vt;
        x[q][t] = (r > i) ? vt : (r == i) ? mk(beta, 0) : xt;
      }
      if (wave == 0 && lane < t) {  // lane j: S(j, t) = v_j^H v_t = conj(v_j(i)) + sc v_j^H x_t
        const int e = 1 + 2 * (NB - 1 - t) + 2 * lane;
        const cplx raw = mk((red[par][0][e] + red[par][1][e]) + (red[par][2][e] + red[par][3][e]),
                            (red[par][0][e + 1] + red[par][1][e + 1]) + (red[par][2][e + 1] + red[par][3][e + 1]));
        cplx sj = conj(mk(piv[par][lane].re, piv[par][lane].im));
        cfma(sj, sc, raw);
        Tl[lane * NB + t] = sj;
      }
      if (tid == 0) {
        taul[t] = tau;
        betal[t] = beta;
      }
    });
    if (tid < kb) {
      D[k0 + tid] = fabs(betal[tid]);
      st(gp(c.qr_tau) + k0 + tid, taul[tid]);
    }
    // ---- zlarft (forward, columnwise) from S: T(t,t) = tau_t, T(0:t, t) = -tau_t T(0:t, 0:t) S(0:t, t);
    // wave 0, lane j keeps row j of T in registers (T(j, l) = 0 for j > l)
    if (wave == 0) {
      cplx trow[NB];
#pragma unroll
      for (int l = 0; l < NB; ++l) trow[l] = mk(0, 0);
      // no branch on t < kb around the LDS reads (that would wait for each read in turn):
      // the S entries and tau of the zero columns past kb are zero, and a select keeps them 0
#pragma unroll
      for (int t = 0; t < NB; ++t) {
        cplx acc = mk(0, 0);
#pragma unroll
        for (int l = 0; l < t; ++l) cfma(acc, trow[l], Tl[l * NB + t]);
        const cplx tt = taul[t];
        const cplx v = (lane < t) ? -(tt * acc) : (lane == t) ? tt : mk(0, 0);
        trow[t] = (t < kb) ? v : mk(0, 0);
      }
      if (lane < NB) {
#pragma unroll
        for (int t = 0; t < NB; ++t) {
          Tl[lane * NB + t] = trow[t];
          st(Tg + lane * NB + t, trow[t]);
        }
      }
    }
    // x back to A (rows >= kw: R above and on the diagonal, reflectors below) and, as the
    // unit lower trapezoid V, to P for the next panel's update
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      gcplx* a = A + (size_t)perm[k0 + min(t, kb - 1)] * n;
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = tid + 256 * q;
        const cplx xv = x[q][t];
        if (r >= k0 && r < n) {
          const cplx pv = (t >= kb || r < k0 + t) ? mk(0, 0) : (r == k0 + t) ? mk(1, 0) : xv;
          P[(size_t)t * ps + r].re = pv.re;
          P[(size_t)t * ps + r].im = pv.im;
        }
        if (t < kb && r >= kw && r < n) {
          a[r].re = xv.re;
          a[r].im = xv.im;
        }
      }
    }  // the group barrier that follows every call publishes P, Tl and A
  };

  // ---- x <- (I - V T^H V^H) x for NB columns held in x (rows >= k0), with V (rows >= k0) in P,
  // this thread's rows of it in pj, and T in Tl: W = V^H x by one butterfly per column, then
  // every wave forms Z = T^H W itself (entry u NB + j on lane (u NB + j) mod 64) and the row
  // updates take Z from scalar registers. V is read from LDS once per panel, not per column.
  cplx pj[RQ][NB];
  auto load_pj = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const int r = tid + 256 * q;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const cplx* src = P + (size_t)j * ps + min(r, n - 1);
        const cplx pv = mk(src->re, src->im);
        pj[q][j] = (r >= k0 && r < n) ? pv : mk(0, 0);
      }
    }
  };
  auto apply_regs = [&]() __attribute__((always_inline)) {
    constexpr int ZE = NB * NB / 64;  // Z entries per lane
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      double v[V];
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = 0.0;
#pragma unroll
      for (int q = 0; q < RQ; ++q)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          v[2 * j] = fma(pj[q][j].re, x[q][u].re, fma(pj[q][j].im, x[q][u].im, v[2 * j]));
          v[2 * j + 1] = fma(pj[q][j].re, x[q][u].im, fma(-pj[q][j].im, x[q][u].re, v[2 * j + 1]));
        }
      wave_reduce_scatter<V>(v);
      if ((lane & ((1 << LS) - 1)) == 0) redW[wave][u][lane >> LS] = v[0];
    }
    __syncthreads();
    cplx zr[ZE];
#pragma unroll
    for (int m = 0; m < ZE; ++m) {
      const int idx = lane + 64 * m, u = idx / NB, j = idx % NB;
      cplx z = mk(0, 0);
#pragma unroll
      for (int l = 0; l < NB; ++l) {
        const cplx wl = mk((redW[0][u][2 * l] + redW[1][u][2 * l]) + (redW[2][u][2 * l] + redW[3][u][2 * l]),
                           (redW[0][u][2 * l + 1] + redW[1][u][2 * l + 1]) +
                               (redW[2][u][2 * l + 1] + redW[3][u][2 * l + 1]));
        cfma_cj(z, Tl[l * NB + j], wl);
      }
      zr[m] = z;
    }
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int idx = u * NB + j;
        const cplx z = read_lane_c(zr[idx / 64], idx % 64);
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
          cplx a = x[q][u];
          a.re = fma(-pj[q][j].re, z.re, fma(pj[q][j].im, z.im, a.re));
          a.im = fma(-pj[q][j].re, z.im, fma(-pj[q][j].im, z.re, a.im));
          x[q][u] = a;
        }
      }
  };
  // rows >= kr of x back to logical columns kc .. kc+kbc-1
  auto store_regs = [&](int kc, int kbc, int kr) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      gcplx* a = A + (size_t)perm[kc + min(t, kbc - 1)] * n;
#pragma unroll
      for (int q = 0; q < RQ; ++q) {
        const int r = tid + 256 * q;
        if (t < kbc && r >= kr && r < n) {
          a[r].re = x[q][t].re;
          a[r].im = x[q][t].im;
        }
      }
    }
  };
  const int ws = W == 1 ? 1 : W - 1, w0 = W == 1 ? 0 : 1;  // trailing workgroups, first one
  // One-panel look-ahead: while every other workgroup applies panel p to the columns beyond
  // panel p+1 (in blocks of NB logical columns, block b to workgroup 1 + b mod (W-1)),
  // workgroup 0 applies it to panel p+1's columns and factors panel p+1, so each panel costs
  // one group barrier and its factorisation overlaps the trailing update. Workgroup 0 keeps
  // V and T of the panel it factored in P and Tl; the others stage them. Iteration p = -1
  // factors panel 0 alone. Each code path has one call site, for the instruction cache.
  for (int p = -1, k1 = 0; k1 < n; ++p, k1 += NB) {  // apply panel p, factor panel p+1 at k1
    const int k0 = k1 - NB;
    if (p >= 0) {
      if (w != 0) {
        stage_panel<NB>(P, A, perm, k0, NB, n, tid, 1, ps);
        for (int e = tid; e < NB * NB; e += blockDim.x) Tl[e] = ld(gp(c.qr_Tf) + (size_t)p * NB * NB + e);
        __syncthreads();
      }
      load_pj(k0);
    }
    // this workgroup's blocks: trailing ones first (kc >= k1 + NB), then, on workgroup 0,
    // panel p+1 itself, which stays in x for the factorisation
    if (p < 0) {
      if (w == 0) load_regs(0, min(NB, n), 0);
    } else {
      for (int kc = (w >= w0) ? k1 + NB + (w - w0) * NB : n;; kc += ws * NB) {
        const bool next = kc >= n;
        if (next && w != 0) break;
        const int kcc = next ? k1 : kc, kbc = min(NB, n - kcc);
        load_regs(kcc, kbc, k0);
        apply_regs();
        if (next) break;
        store_regs(kcc, kbc, k0);
        __syncthreads();  // redW is reused by the next block
      }
    }
    if (w == 0) factor_regs(k1, p + 1, p >= 0 ? k0 : 0);
    group_sync(g);
    if (group_failed(g)) return;
  }
  if (w == 0) {
    for (int k = tid; k < n; k += blockDim.x) {
      gp(c.qr_perm)[k] = perm[k];
      gp(c.qr_lpos)[k] = lpos[k];
    }
  }
}

// k_qr_solve / k_form_Q_blocked: a workgroup owns CB columns in LDS, CB / 4 per wave, so every V
// entry read from LDS serves CB / 4 columns.
//
// x <- (I - V op(T) V^H) x for this wave's CPW columns xc + (jl0 + c) n (rows >= k0); V [NB][n]
// and T (Tl[j * NB + l] = T(j, l)) in LDS; op = T^H (ADJ, applying Q^H) or T (applying Q).
template <int NB, int CB, bool ADJ>
__device__ inline void apply_panel_cols(cplx* xc, const cplx* V, const cplx* Tl, int n, int k0, int jl0, int ncol,
                                        int lane) {
  constexpr int CPW = CB / 4;
  cplx wv[CPW][NB];
#pragma unroll
  for (int c = 0; c < CPW; ++c)
#pragma unroll
    for (int j = 0; j < NB; ++j) wv[c][j] = mk(0, 0);
  for (int k = k0 + lane; k < n; k += 64) {
    cplx pj[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) pj[j] = V[(size_t)j * n + k];
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
      const cplx ak = xc[(size_t)(jl0 + c) * n + k];
#pragma unroll
      for (int j = 0; j < NB; ++j) cfma_cj(wv[c][j], pj[j], ak);
    }
  }
#pragma unroll
  for (int c = 0; c < CPW; ++c) wave_sum_many<NB>(wv[c]);
  // z = op(T) w: lane j < NB forms z_j of every column, then every lane reads them
  const int jz = lane & (NB - 1);
  cplx z[CPW][NB];
#pragma unroll
  for (int c = 0; c < CPW; ++c) {
    cplx zl = mk(0, 0);
#pragma unroll
    for (int l = 0; l < NB; ++l) {
      if (ADJ)
        cfma_cj(zl, Tl[l * NB + jz], wv[c][l]);
      else
        cfma(zl, Tl[jz * NB + l], wv[c][l]);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) z[c][j] = read_lane_c(zl, j);
  }
  if (jl0 < ncol) {  // wave-uniform; columns past ncol of the group are scratch
    for (int k = k0 + lane; k < n; k += 64) {
      cplx pj[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) pj[j] = V[(size_t)j * n + k];
#pragma unroll
      for (int c = 0; c < CPW; ++c) {
        cplx ak = xc[(size_t)(jl0 + c) * n + k];
#pragma unroll
        for (int j = 0; j < NB; ++j) ak = ak - pj[j] * z[c][j];
        xc[(size_t)(jl0 + c) * n + k] = ak;
      }
    }
  }
}

// B <- R^-1 Q^H B for a matrix factored by k_qr_blocked without pre-pivoting (Ar holds R and
// the reflectors, qr_tau / qr_Tf the rest). Every right-hand side is independent: each
// workgroup owns CB columns of B in LDS, applies the panels' Q_p^H in order, then
// back-substitutes with R; no synchronisation between workgroups. (16-column panels; 8-column
// ones take k_qr_solve_rows.)
template <int NB, int CB>
__global__ __launch_bounds__(256) void k_qr_solve(const ChainDesc* chains, MatRef Ar, MatRef Br) {
  int bx, by;
  xcd_block(bx, by);
  const ChainDesc& c = chains[by];
  const int n = c.n;
  const int j0 = bx * CB;
  if (j0 >= n) return;
  const int ncol = min(CB, n - j0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int jl0 = wave * (CB / 4);
  const gcplx* A = gp(matptr(c, Ar));
  gcplx* B = gp(matptr(c, Br));
  extern __shared__ double smem[];
  cplx* bc = reinterpret_cast<cplx*>(smem);  // [CB][n]
  cplx* V = bc + (size_t)CB * n;              // [NB][n]
  __shared__ cplx Tl[NB * NB];
  __shared__ cplx Rd[16 * 16];
  for (int r = tid; r < n; r += 256) {
    cplx v[CB];
#pragma unroll
    for (int q = 0; q < CB; ++q) {
      const gcplx* src = B + (size_t)(j0 + min(q, ncol - 1)) * n + r;
      v[q] = mk(src->re, src->im);  // (a whole-struct copy here is lowered through a stack slot)
    }
#pragma unroll
    for (int q = 0; q < CB; ++q) bc[(size_t)q * n + r] = v[q];
  }
  for (int k0 = 0, p = 0; k0 < n; k0 += NB, ++p) {
    const int kb = min(NB, n - k0);
    __syncthreads();
    stage_panel<NB>(V, A, nullptr, k0, kb, n, tid, 1);  // columns >= kb zero-filled
    for (int e = tid; e < NB * NB; e += blockDim.x) Tl[e] = ld(gp(c.qr_Tf) + (size_t)p * NB * NB + e);
    __syncthreads();
    apply_panel_cols<NB, CB, true>(bc, V, Tl, n, k0, jl0, ncol, lane);
  }
  // back substitution R y = z in blocks of 16 rows from the bottom: wave q < CB solves the
  // 16 x 16 diagonal block for column q (lane r holds row lo + r), then every thread takes
  // rows r < lo and subtracts the block's contribution for all CB columns, reading R's
  // block column once (sixteen loads in flight per row)
  for (int hi = n; hi > 0; hi -= 16) {
    const int lo = max(0, hi - 16), bs = hi - lo;
    __syncthreads();
    {
      const int kk = tid >> 4, rr = tid & 15;
      Rd[tid] = (kk < bs && rr < bs) ? ld(A + (size_t)(lo + kk) * n + lo + rr) : mk(0, 0);  // Rd[kk*16+rr] = R(lo+rr, lo+kk)
    }
    __syncthreads();
    for (int q = wave; q < ncol; q += 4) {  // wave-uniform: the 16 x 16 diagonal solve of column q
      cplx* y = bc + (size_t)q * n;
      const int r = lo + (lane & 15);
      cplx zr = (lane < bs) ? y[r] : mk(0, 0);
      for (int k = bs - 1; k >= 0; --k) {
        const cplx yk = shfl_c(zr, k) * cinv(Rd[k * 16 + k]);
        if (lane < k) zr = zr - Rd[k * 16 + (lane & 15)] * yk;
        if (lane == k) zr = yk;
      }
      if (lane < bs) y[r] = zr;
    }
    __syncthreads();
    for (int r = tid; r < lo; r += 256) {
      cplx rv[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) rv[k] = ld(A + (size_t)(lo + min(k, bs - 1)) * n + r);
#pragma unroll
      for (int q = 0; q < CB; ++q) {
        cplx* y = bc + (size_t)q * n;
        cplx acc = y[r];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const cplx yk = y[min(lo + k, n - 1)];
          acc = acc - rv[k] * ((k < bs) ? yk : mk(0, 0));
        }
        y[r] = acc;
      }
    }
  }
  __syncthreads();
  for (int r = tid; r < n; r += 256) {
    cplx v[CB];
#pragma unroll
    for (int q = 0; q < CB; ++q) v[q] = bc[(size_t)q * n + r];
#pragma unroll
    for (int q = 0; q < CB; ++q)
      if (q < ncol) {
        gcplx* d = B + (size_t)(j0 + q) * n + r;
        d->re = v[q].re;
        d->im = v[q].im;
      }
  }
}

// Q = Q_1 Q_2 ... Q_P of a factorisation by k_qr_blocked, Q_p = I - V_p T_p V_p^H
// (zungqr's result, formed from the compact-WY panels instead of one reflector at a time).
// Each workgroup owns CB columns of Q in LDS, starting from the identity, and applies the
// panels from the last one that reaches its columns down to the first; the waves split as
// in k_qr_solve. Reflector k lives in physical column qr_perm[k] below its diagonal.
template <int NB, int CB>
__global__ __launch_bounds__(256) void k_form_Q_blocked(const ChainDesc* chains, MatRef Ar, MatRef Qr) {
  int bx, by;
  xcd_block(bx, by);
  const ChainDesc& c = chains[by];
  const int n = c.n;
  const int j0 = bx * CB;
  if (j0 >= n) return;
  const int ncol = min(CB, n - j0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int jl0 = wave * (CB / 4);
  const gcplx* A = gp(matptr(c, Ar));
  gcplx* Q = gp(matptr(c, Qr));
  extern __shared__ double smem[];
  cplx* xc = reinterpret_cast<cplx*>(smem);  // [CB][n]
  cplx* V = xc + (size_t)CB * n;              // [NB][n]
  __shared__ cplx Tl[NB * NB];
  for (int r = tid; r < n; r += 256)
#pragma unroll
    for (int q = 0; q < CB; ++q) {
      xc[(size_t)q * n + r].re = (r == j0 + q) ? 1.0 : 0.0;
      xc[(size_t)q * n + r].im = 0.0;
    }
  const int jmax = j0 + ncol - 1;  // panels starting beyond it leave these columns alone
  for (int p = jmax / NB; p >= 0; --p) {
    const int k0 = p * NB, kb = min(NB, n - k0);
    __syncthreads();
    stage_panel<NB>(V, A, c.qr_perm, k0, kb, n, tid, 1);  // columns >= kb zero-filled
    for (int e = tid; e < NB * NB; e += blockDim.x) Tl[e] = ld(gp(c.qr_Tf) + (size_t)p * NB * NB + e);
    __syncthreads();
    apply_panel_cols<NB, CB, false>(xc, V, Tl, n, k0, jl0, ncol, lane);
  }
  __syncthreads();
  for (int r = tid; r < n; r += 256) {
    cplx v[CB];
#pragma unroll
    for (int q = 0; q < CB; ++q) v[q] = xc[(size_t)q * n + r];
#pragma unroll
    for (int q = 0; q < CB; ++q)
      if (q < ncol) {
        gcplx* d = Q + (size_t)(j0 + q) * n + r;
        d->re = v[q].re;
        d->im = v[q].im;
      }
  }
}

// ---------------------------------------------------------------------------
// Solve and Q formation with the columns in registers (few chains per launch).
//
// A workgroup owns four columns, thread t their rows t + 256 q (RQ = rows per thread). A panel's
// reflectors go from memory straight into the registers of the threads that own their rows and
// serve both products there, so each entry is read once per workgroup and never passes LDS:
// W = V^H X is 32 sums per wave by one butterfly, the four waves' sums meet in LDS (one barrier
// per panel, two buffers), every wave forms Z = op(T) W by itself (lane = column, reflector and
// half of the sum). The kernels before it staged V in LDS (one column per workgroup at n > 640,
// where V alone takes 131 KB). Bound by the chain of a panel: V's latency, the butterfly, the
// barrier. n = 1024: solve 4.07 -> 1.11 ms, Q 2.49 -> 0.70 ms; n = 400: 0.419 -> 0.293 and 0.189 ->
// 0.189 ms; n = 256: 0.220 -> 0.160 and 0.098 -> 0.098 ms; n = 576, Q of two chains: 0.57 -> 0.52 ms.
// ---------------------------------------------------------------------------
constexpr int kRowCols = 4;

struct RowsShared {
  double part[2][4][64];  // per wave: the 32 complex sums
  cplx z[4][32];          // per wave: Z
};

template <int RQ, bool ADJ>
__device__ inline void apply_panel_rows(cplx (&x)[RQ][kRowCols], const gcplx* A, const gcplx* Tf, const int* perm,
                                        int p, int n, RowsShared& sh) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k0 = 8 * p;
  cplx v[RQ][8];
#pragma unroll
  for (int q = 0; q < RQ; ++q) {
    const int r = tid + 256 * q, rr = min(r, n - 1);
    if (256 * q + 255 >= k0) {  // (uniform) some rows at or below the diagonal
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = min(k0 + j, n - 1);
        v[q][j] = ld(A + (size_t)(perm ? perm[k] : k) * n + rr);
      }
    }
  }
  // this lane's half of a row of op(T)
  const int zc = (lane >> 3) & 3, zj = lane & 7, zh = lane >> 5;
  cplx t[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) t[u] = ld(Tf + 64 * p + (ADJ ? (4 * zh + u) * 8 + zj : zj * 8 + 4 * zh + u));
  double w[64];
#pragma unroll
  for (int e = 0; e < 64; ++e) w[e] = 0.0;
#pragma unroll
  for (int q = 0; q < RQ; ++q) {
    const int r = tid + 256 * q;
    if (256 * q + 255 >= k0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int k = k0 + j;
        const bool below = r > k && r < n && k < n;
        v[q][j].re = below ? v[q][j].re : (r == k && k < n) ? 1.0 : 0.0;
        v[q][j].im = below ? v[q][j].im : 0.0;
#pragma unroll
        for (int c = 0; c < kRowCols; ++c) {
          cplx s = mk(w[2 * (8 * c + j)], w[2 * (8 * c + j) + 1]);
          cfma_cj(s, v[q][j], x[q][c]);
          w[2 * (8 * c + j)] = s.re;
          w[2 * (8 * c + j) + 1] = s.im;
        }
      }
    }
  }
  wave_reduce_scatter<64>(w);
  const int buf = p & 1;
  sh.part[buf][wave][lane] = w[0];
  __syncthreads();
  cplx z = mk(0, 0);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int e = 2 * (8 * zc + 4 * zh + u);
    cplx s = mk(0, 0);
#pragma unroll
    for (int g = 0; g < 4; ++g) s += mk(sh.part[buf][g][e], sh.part[buf][g][e + 1]);
    if (ADJ)
      cfma_cj(z, t[u], s);
    else
      cfma(z, t[u], s);
  }
  z.re += __shfl_xor(z.re, 32, 64);
  z.im += __shfl_xor(z.im, 32, 64);
  if (lane < 32) {
    sh.z[wave][lane].re = z.re;
    sh.z[wave][lane].im = z.im;
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
  for (int c = 0; c < kRowCols; ++c) {
    cplx zz[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) zz[j] = sh.z[wave][8 * c + j];
#pragma unroll
    for (int q = 0; q < RQ; ++q)
      if (256 * q + 255 >= k0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) cfma(x[q][c], -v[q][j], zz[j]);
      }
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // Z read before the next panel's
}

template <int RQ>
__global__ __launch_bounds__(256) void k_form_Q_rows(const ChainDesc* chains, MatRef Ar, MatRef Qr) {
  int bx, by;
  xcd_block(bx, by);
  const ChainDesc& c = chains[by];
  const int n = c.n, j0 = bx * kRowCols, tid = threadIdx.x;
  if (j0 >= n) return;
  const int ncol = min(kRowCols, n - j0);
  const gcplx* A = gp(matptr(c, Ar));
  gcplx* Q = gp(matptr(c, Qr));
  __shared__ RowsShared sh;
  __shared__ int perm[kQrMaxN];
  for (int k = tid; k < n; k += 256) perm[k] = c.qr_perm[k];
  __syncthreads();
  cplx x[RQ][kRowCols];
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int u = 0; u < kRowCols; ++u) x[q][u] = mk(tid + 256 * q == j0 + u ? 1.0 : 0.0, 0.0);
  for (int p = (j0 + ncol - 1) / 8; p >= 0; --p)  // panels that start beyond the columns leave them alone
    apply_panel_rows<RQ, false>(x, A, gp(c.qr_Tf), perm, p, n, sh);
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int u = 0; u < kRowCols; ++u)
      if (tid + 256 * q < n && u < ncol) st(Q + (size_t)(j0 + u) * n + tid + 256 * q, x[q][u]);
}

template <int RQ>
__global__ __launch_bounds__(256) void k_qr_solve_rows(const ChainDesc* chains, MatRef Ar, MatRef Br) {
  int bx, by;
  xcd_block(bx, by);
  const ChainDesc& c = chains[by];
  const int n = c.n, j0 = bx * kRowCols, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (j0 >= n) return;
  const int ncol = min(kRowCols, n - j0);
  const gcplx* A = gp(matptr(c, Ar));
  gcplx* B = gp(matptr(c, Br));
  __shared__ RowsShared sh;
  __shared__ cplx Rd[16 * 17], Y[kRowCols][16], S[kRowCols][16];
  cplx x[RQ][kRowCols];
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int u = 0; u < kRowCols; ++u)
      x[q][u] = ld(B + (size_t)(j0 + min(u, ncol - 1)) * n + min(tid + 256 * q, n - 1));
  for (int p = 0; 8 * p < n; ++p) apply_panel_rows<RQ, true>(x, A, gp(c.qr_Tf), nullptr, p, n, sh);
  // back substitution in aligned blocks of 16 rows from the bottom: wave u solves the 16 x 16
  // diagonal block for column u (lane = row), then every thread takes its rows above
  for (int hi = n; hi > 0; hi = (hi - 1) & ~15) {
    const int lo = (hi - 1) & ~15, bs = hi - lo, qb = lo >> 8;
    {
      const int kk = tid >> 4, rr = tid & 15;
      const cplx v = ld(A + (size_t)min(lo + kk, n - 1) * n + min(lo + rr, n - 1));
      Rd[kk * 17 + rr].re = v.re;  // R(lo + rr, lo + kk)
      Rd[kk * 17 + rr].im = v.im;
    }
    if (((tid ^ lo) & 0xF0) == 0) {  // the sixteen threads whose rows are the block's
#pragma unroll
      for (int q = 0; q < RQ; ++q)
        if (q == qb) {
#pragma unroll
          for (int u = 0; u < kRowCols; ++u) {
            Y[u][tid & 15].re = x[q][u].re;
            Y[u][tid & 15].im = x[q][u].im;
          }
        }
    }
    __syncthreads();
    {
      const int r = lane & 15;
      cplx zr = Y[wave][r];
      const cplx dv = cinv(Rd[min(r, bs - 1) * 18]);
      for (int k = bs - 1; k >= 0; --k) {
        const cplx yk = read_lane_c(zr, k) * read_lane_c(dv, k);
        const cplx rk = Rd[k * 17 + r];
        if (r < k) zr = zr - rk * yk;
        if (r == k) zr = yk;
      }
      if (lane < 16) {
        S[wave][r].re = r < bs ? zr.re : 0.0;
        S[wave][r].im = r < bs ? zr.im : 0.0;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RQ; ++q) {
      const int r = tid + 256 * q;
      if (256 * q < lo) {
        cplx rv[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) rv[k] = ld(A + (size_t)min(lo + k, n - 1) * n + min(r, n - 1));
        if (r < lo) {
#pragma unroll
          for (int u = 0; u < kRowCols; ++u)
#pragma unroll
            for (int k = 0; k < 16; ++k) cfma(x[q][u], -rv[k], S[u][k]);
        }
      }
      if (q == qb && r >= lo && r < hi) {
#pragma unroll
        for (int u = 0; u < kRowCols; ++u) x[q][u] = mk(S[u][tid & 15].re, S[u][tid & 15].im);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < RQ; ++q)
#pragma unroll
    for (int u = 0; u < kRowCols; ++u)
      if (tid + 256 * q < n && u < ncol) st(B + (size_t)(j0 + u) * n + tid + 256 * q, x[q][u]);
}

// rows per thread by size
template <class K>
hipError_t launch_rows(K k1, K k2, K k3, K k4, hipStream_t s, const ChainDesc* chains, int nchains, int nmax, MatRef A,
                       MatRef X) {
  const K fn = nmax <= 256 ? k1 : nmax <= 512 ? k2 : nmax <= 768 ? k3 : k4;
  hipLaunchKernelGGL(fn, dim3((nmax + kRowCols - 1) / kRowCols, nchains), dim3(256), 0, s, chains, A, X);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Panel application on the FP64 matrix cores for LDS-resident column blocks (k_qr_solve_mfma,
// k_form_Q_mfma). The workgroup owns CB <= 16 columns of X (one 16-column MFMA tile) and
// applies one 8-column compact-WY panel, X <- (I - V op(T) V^H) X on the rows >= k0:
//   W = V^H X (8 x CB): v_mfma_f64_16x16x4 with A(i, k) = conj V(r, i) (rows 8..15 of the
//     tile zero) and B(k, j) = X(r, j), the rows split into four contiguous ranges, one per
//     wave; waves 1-3 leave their partial W in LDS, wave 0 adds them, forms Z = op(T) W with
//     the vector units and leaves Z in LDS;
//   X -= V Z: 16-row tiles of X spread over the waves, A(i, k) = V(r0 + i, k), B(k, j) =
//     Z(k, j), two k-steps.
// A complex product is four real MFMAs. Lane layout of v_mfma_f64_16x16x4: A(i, k) and
// B(k, j) on lane i + 16 k (resp. j + 16 k); D(i, j) element v on lane j + 16 (i - 4 v).
// LDS: X [CB][ld], V [8][ld] (unit lower trapezoid from stage_panel), 3 x 8 x 16 scratch.
// ---------------------------------------------------------------------------
constexpr int kMfmaScratch = 3 * 8 * 16;  // complex entries of the panel scratch

template <int CB, bool ADJ>
__device__ inline void apply_panel_mfma(cplx* xc, const cplx* V, const cplx* Tl, cplx* scr, int n, int cs,
                                        int k0) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int vi = min(li, 7), xj = min(li, CB - 1);
  const int nst = (n - k0) >> 2;  // n - k0 is a multiple of 4
  const int sa = (nst * wave) >> 2, sb = (nst * (wave + 1)) >> 2;
  v4d wr = {0.0, 0.0, 0.0, 0.0}, wi = {0.0, 0.0, 0.0, 0.0};
  for (int st = sa; st < sb; ++st) {
    const int r = k0 + 4 * st + lk;
    const cplx v = V[(size_t)vi * cs + r];
    const cplx x = xc[(size_t)xj * cs + r];
    const double vr = li < 8 ? v.re : 0.0, vm = li < 8 ? v.im : 0.0;
    const double xr = li < CB ? x.re : 0.0, xm = li < CB ? x.im : 0.0;
    // W += V^H X: re += Vr Xr + Vi Xi, im += Vr Xi - Vi Xr
    wr = mfma4(vr, xr, wr);
    wi = mfma4(vr, xm, wi);
    wr = mfma4(vm, xm, wr);
    wi = mfma4(-vm, xr, wi);
  }
  // lane (li, lk) holds W(lk, li) (element 0) and W(lk + 4, li) (element 1)
  if (wave > 0) {
    cplx* q = scr + (wave - 1) * 128;
    q[lk * 16 + li] = mk(wr[0], wi[0]);
    q[(lk + 4) * 16 + li] = mk(wr[1], wi[1]);
  }
  __syncthreads();
  if (wave == 0) {
    cplx w0 = mk(wr[0], wi[0]), w1 = mk(wr[1], wi[1]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      w0 += scr[q * 128 + lk * 16 + li];
      w1 += scr[q * 128 + (lk + 4) * 16 + li];
    }
    // the full W over wave 1's partial (each lane rewrites only the entries it read)
    scr[lk * 16 + li] = w0;
    scr[(lk + 4) * 16 + li] = w1;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    cplx z0 = mk(0, 0), z1 = mk(0, 0);
#pragma unroll
    for (int l = 0; l < 8; ++l) {
      const cplx wl = scr[l * 16 + li];
      if (ADJ) {  // Z = T^H W
        cfma_cj(z0, Tl[l * 8 + lk], wl);
        cfma_cj(z1, Tl[l * 8 + lk + 4], wl);
      } else {  // Z = T W
        cfma(z0, Tl[lk * 8 + l], wl);
        cfma(z1, Tl[(lk + 4) * 8 + l], wl);
      }
    }
    scr[128 + lk * 16 + li] = z0;
    scr[128 + (lk + 4) * 16 + li] = z1;
  }
  __syncthreads();
  const cplx* Zs = scr + 128;
  const int nrb = (n - k0 + 15) >> 4;
  for (int rb = wave; rb < nrb; rb += 4) {
    const int r0 = k0 + 16 * rb;
    v4d dr, di;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int row = min(r0 + lk + 4 * v, n - 1);
      const cplx x = xc[(size_t)xj * cs + row];
      dr[v] = x.re;
      di[v] = x.im;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int ra = r0 + li;
      const cplx a0 = V[(size_t)(4 * ks + lk) * cs + min(ra, n - 1)];
      const double ar = ra < n ? a0.re : 0.0, am = ra < n ? a0.im : 0.0;
      const cplx z = Zs[(4 * ks + lk) * 16 + li];
      // X -= V Z: re += -Vr Zr + Vi Zi, im += -Vr Zi - Vi Zr
      dr = mfma4(-ar, z.re, dr);
      di = mfma4(-ar, z.im, di);
      dr = mfma4(am, z.im, dr);
      di = mfma4(-am, z.re, di);
    }
    if (li < CB) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = r0 + lk + 4 * v;
        if (row < n) xc[(size_t)li * cs + row] = mk(dr[v], di[v]);
      }
    }
  }
}

// k_qr_solve on the matrix cores: B <- R^-1 Q^H B with CB columns per workgroup. The panels'
// Q_p^H as in apply_panel_mfma; the back substitution in blocks of 16 rows from the bottom:
// each wave solves the 16 x 16 diagonal block for four columns at once (lane = row + 16 x
// column; the block's inverse diagonal precomputed once), then the rows above take the
// block's contribution as MFMA tiles, R(r, lo:hi) y(lo:hi, :) (K = 16).
template <int CB>
__global__ __launch_bounds__(256) void k_qr_solve_mfma(const ChainDesc* chains, MatRef Ar, MatRef Br, int cs, int nlo, int nhi) {
  int bx, by;
  xcd_block(bx, by);
  const ChainDesc& c = chains[by];
  const int n = c.n;
  const int j0 = bx * CB;
  if (j0 >= n || n <= nlo || n > nhi) return;  // outside this launch's size class
  const int ncol = min(CB, n - j0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = lane >> 4;
  const gcplx* A = gp(matptr(c, Ar));
  gcplx* B = gp(matptr(c, Br));
  extern __shared__ double smem[];
  cplx* xc = reinterpret_cast<cplx*>(smem);  // [CB][cs]
  cplx* V = xc + (size_t)CB * cs;             // [8][cs]; the back substitution's diagonal block
  cplx* scr = V + (size_t)8 * cs;             // panel scratch
  __shared__ cplx Tl[64];
  for (int r = tid; r < n; r += 256) {
    cplx v[CB];
#pragma unroll
    for (int q = 0; q < CB; ++q) v[q] = ld(B + (size_t)(j0 + min(q, ncol - 1)) * n + r);
#pragma unroll
    for (int q = 0; q < CB; ++q) {
      xc[(size_t)q * cs + r].re = v[q].re;  // (a whole-struct copy from a register array is
      xc[(size_t)q * cs + r].im = v[q].im;  // lowered through a stack slot)
    }
  }
  for (int k0 = 0, p = 0; k0 < n; k0 += 8, ++p) {
    const int kb = min(8, n - k0);
    __syncthreads();
    stage_panel<8>(V, A, nullptr, k0, kb, n, tid, 1, cs);  // columns >= kb zero-filled
    if (tid < 64) Tl[tid] = ld(gp(c.qr_Tf) + (size_t)p * 64 + tid);
    __syncthreads();
    apply_panel_mfma<CB, true>(xc, V, Tl, scr, n, cs, k0);
  }
  cplx* Rd = V;        // [16][16]: Rd[kk * 16 + rr] = R(lo + rr, lo + kk)
  cplx* Ri = V + 256;  // [16]: 1 / R(lo + k, lo + k)
  const int xj = min(li, CB - 1);
  for (int hi = n; hi > 0; hi -= 16) {
    const int lo = max(0, hi - 16), bs = hi - lo;
    __syncthreads();
    {
      const int kk = tid >> 4, rr = tid & 15;
      Rd[tid] = (kk < bs && rr < bs) ? ld(A + (size_t)(lo + kk) * n + lo + rr) : mk(0, 0);
      if (tid < 16) Ri[tid] = tid < bs ? cinv(ld(A + (size_t)(lo + tid) * n + lo + tid)) : mk(0, 0);
    }
    __syncthreads();
    {  // wave w: columns w + 4 lk, lane row li
      const int col = wave + 4 * lk;
      cplx* y = xc + (size_t)min(col, CB - 1) * cs;
      cplx zr = li < bs ? y[lo + li] : mk(0, 0);
      for (int k = bs - 1; k >= 0; --k) {
        const cplx yk = shfl_c(zr, (lane & 48) + k) * Ri[k];
        if (li < k) zr = zr - Rd[k * 16 + li] * yk;
        if (li == k) zr = yk;
      }
      if (col < CB && li < bs) y[lo + li] = zr;
    }
    __syncthreads();
    const int nrb = (lo + 15) >> 4;
    for (int rb = wave; rb < nrb; rb += 4) {
      const int r0 = rb * 16;
      v4d dr, di;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const cplx x = xc[(size_t)xj * cs + min(r0 + lk + 4 * v, n - 1)];
        dr[v] = x.re;
        di[v] = x.im;
      }
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int kk = 4 * ks + lk, ra = r0 + li;
        const cplx a0 = ld(A + (size_t)(lo + min(kk, bs - 1)) * n + min(ra, n - 1));
        const cplx y0 = xc[(size_t)xj * cs + lo + min(kk, bs - 1)];
        const bool ok = kk < bs && ra < lo;
        const double ar = ok ? a0.re : 0.0, am = ok ? a0.im : 0.0;
        const double yr = kk < bs ? y0.re : 0.0, ym = kk < bs ? y0.im : 0.0;
        // z -= R y
        dr = mfma4(-ar, yr, dr);
        di = mfma4(-ar, ym, di);
        dr = mfma4(am, ym, dr);
        di = mfma4(-am, yr, di);
      }
      if (li < CB) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = r0 + lk + 4 * v;
          if (row < lo) xc[(size_t)li * cs + row] = mk(dr[v], di[v]);
        }
      }
    }
  }
  __syncthreads();
  for (int r = tid; r < n; r += 256) {
    cplx v[CB];
#pragma unroll
    for (int q = 0; q < CB; ++q) v[q] = xc[(size_t)q * cs + r];
#pragma unroll
    for (int q = 0; q < CB; ++q)
      if (q < ncol) st(B + (size_t)(j0 + q) * n + r, v[q]);
  }
}

// k_form_Q_blocked on the matrix cores: CB columns of Q per workgroup from the identity, the
// panels from the last one that reaches them down to the first (Q_p = I - V_p T_p V_p^H).
template <int CB>
__global__ __launch_bounds__(256) void k_form_Q_mfma(const ChainDesc* chains, MatRef Ar, MatRef Qr, int cs, int nlo, int nhi) {
  int bx, by;
  xcd_block(bx, by);
  const ChainDesc& c = chains[by];
  const int n = c.n;
  const int j0 = bx * CB;
  if (j0 >= n || n <= nlo || n > nhi) return;  // outside this launch's size class
  const int ncol = min(CB, n - j0);
  const int tid = threadIdx.x;
  const gcplx* A = gp(matptr(c, Ar));
  gcplx* Q = gp(matptr(c, Qr));
  extern __shared__ double smem[];
  cplx* xc = reinterpret_cast<cplx*>(smem);  // [CB][cs]
  cplx* V = xc + (size_t)CB * cs;             // [8][cs]
  cplx* scr = V + (size_t)8 * cs;
  __shared__ cplx Tl[64];
  for (int e = tid; e < CB * n; e += 256) {
    const int q = e / n, r = e - q * n;
    xc[(size_t)q * cs + r] = mk(r == j0 + q ? 1.0 : 0.0, 0.0);
  }
  const int jmax = j0 + ncol - 1;  // panels starting beyond it leave these columns alone
  for (int p = jmax / 8; p >= 0; --p) {
    const int k0 = p * 8, kb = min(8, n - k0);
    __syncthreads();
    stage_panel<8>(V, A, c.qr_perm, k0, kb, n, tid, 1, cs);  // columns >= kb zero-filled
    if (tid < 64) Tl[tid] = ld(gp(c.qr_Tf) + (size_t)p * 64 + tid);
    __syncthreads();
    apply_panel_mfma<CB, false>(xc, V, Tl, scr, n, cs, k0);
  }
  __syncthreads();
  for (int e = tid; e < ncol * n; e += 256) {
    const int q = e / n, r = e - q * n;
    st(Q + (size_t)j0 * n + e, xc[(size_t)q * cs + r]);
  }
}

// columns per workgroup of the matrix-core solve and Q formation at this size (0: the vector
// kernels): 16 while X, V and the scratch fit the LDS (n <= 400), 8 up to n = 576
inline int mfma_cols(int nmax) { return nmax <= 400 ? 16 : nmax <= 576 ? 8 : 0; }
inline size_t mfma_lds(int nmax, int cb) {
  return ((size_t)(cb + 8) * mfma_ld(nmax) + kMfmaScratch) * sizeof(cplx);
}

// chain counts from which solve and Q formation take the matrix-core kernels (16 or 8 columns
// per workgroup); with fewer, the latency of the panel sequence counts and four columns in
// registers finish sooner
constexpr int kWideColChains = 8;

// default panel width: 8 (the register-resident panel keeps nb x rows-per-thread values per
// thread; at nb = 16 the per-column chain is longer and the kernel spills)
int qr_panel_width(int nmax) {
  (void)nmax;
  return 8;
}

static hipError_t launch_qr_kernel(const void* fn, size_t lds, hipStream_t s, const ChainDesc* chains, int nchains,
                                   int ps, MatRef A, VecRef D, int prepivot, int wg, const int* bmap, int nblocks) {
  {
    hipError_t e = ensure_dynamic_lds(fn, lds);
    if (e != hipSuccess) return e;
  }
  void* args[] = {(void*)&chains, (void*)&A, (void*)&D, (void*)&prepivot, (void*)&ps, (void*)&bmap};
  const dim3 grid = bmap ? dim3(nblocks, 1) : dim3(wg, nchains);
  hipError_t e = hipLaunchCooperativeKernel(fn, grid, dim3(256), args, lds, s);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

hipError_t launch_qr_blocked(hipStream_t s, const ChainDesc* chains, int nchains, int nmax, MatRef A, VecRef D,
                             int prepivot, int wg, int nb, const int* bmap, int nblocks) {
  if (nmax > kQrMaxN) return hipErrorInvalidValue;
  if (nb == 0) nb = qr_panel_width(nmax);
  int ps = mfma_ld(nmax);
  if (nb == 16 && nmax <= 512)
    return launch_qr_kernel((const void*)k_qr_blocked<16, 2>, (size_t)16 * ps * sizeof(cplx), s, chains, nchains, ps, A,
                            D, prepivot, wg, bmap, nblocks);
  if (nb != 8) return hipErrorInvalidValue;
  // (a block map gives the chains of each size their workgroups, more for the larger)
  const bool wide = nmax > 512 && !bmap && (wg == 1 || nmax >= 128 * (wg - 1));
  const void* fn = nmax <= 256   ? (const void*)k_qr_pipe<1, false>
                   : nmax <= 512 ? (const void*)k_qr_pipe<2, false>
                   : nmax <= 768 ? (wide ? (const void*)k_qr_pipe<3, true> : (const void*)k_qr_pipe<3, false>)
                   : wide        ? (const void*)k_qr_pipe<4, true>
                                 : (const void*)k_qr_pipe<4, false>;
  ps = mfma_ld(nmax + 16);
  return launch_qr_kernel(fn, ((size_t)8 * ps + 512) * sizeof(cplx), s, chains, nchains, ps, A, D, prepivot, wg, bmap,
                          nblocks);
}

template <int NB, int CB>
hipError_t launch_qr_solve_nb(hipStream_t s, const ChainDesc* chains, int nchains, int nmax, MatRef A, MatRef B) {
  const size_t lds = (size_t)(CB + NB) * nmax * sizeof(cplx);
  {
    hipError_t e = ensure_dynamic_lds((const void*)k_qr_solve<NB, CB>, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_qr_solve<NB, CB>), dim3((nmax + CB - 1) / CB, nchains), dim3(256), lds, s, chains, A, B);
  return hipGetLastError();
}

template <int NB, int CB>
hipError_t launch_form_Q_blocked_nb(hipStream_t s, const ChainDesc* chains, int nchains, int nmax, MatRef A,
                                    MatRef Q) {
  const size_t lds = (size_t)(CB + NB) * nmax * sizeof(cplx);
  {
    hipError_t e = ensure_dynamic_lds((const void*)k_form_Q_blocked<NB, CB>, lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((k_form_Q_blocked<NB, CB>), dim3((nmax + CB - 1) / CB, nchains), dim3(256), lds, s, chains, A,
                     Q);
  return hipGetLastError();
}

template <int CB>
hipError_t launch_mfma_kernel(const void* fn, hipStream_t s, int nchains, int nmax, const ChainDesc* chains, MatRef A,
                              MatRef X, int nlo, int nhi) {
  const size_t lds = mfma_lds(nmax, CB);
  {
    hipError_t e = ensure_dynamic_lds(fn, lds);
    if (e != hipSuccess) return e;
  }
  int cs = mfma_ld(nmax);
  void* args[] = {(void*)&chains, (void*)&A, (void*)&X, (void*)&cs, (void*)&nlo, (void*)&nhi};
  hipError_t e = hipLaunchKernel(fn, dim3((nmax + CB - 1) / CB, nchains), dim3(256), args, lds, s);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

// the matrix-core solve / Q formation over chains up to nmax: chains with n <= 400 take 16
// columns per workgroup, larger ones 8 (two launches when the sizes are mixed; the chains of
// the other class return at once)
template <class F16, class F8>
hipError_t launch_mfma_classes(F16 k16, F8 k8, hipStream_t s, int nchains, int nmax, const ChainDesc* chains, MatRef A,
                               MatRef X) {
  if (nmax <= 400) return launch_mfma_kernel<16>((const void*)k16, s, nchains, nmax, chains, A, X, 0, nmax);
  hipError_t e = launch_mfma_kernel<16>((const void*)k16, s, nchains, 400, chains, A, X, 0, 400);
  if (e != hipSuccess) return e;
  return launch_mfma_kernel<8>((const void*)k8, s, nchains, nmax, chains, A, X, 400, nmax);
}

hipError_t launch_form_Q_blocked(hipStream_t s, const ChainDesc* chains, int nchains, int nmax, MatRef A, MatRef Q,
                                 int nb) {
  if (nmax > kQrMaxN || nmax < 16) return hipErrorInvalidValue;
  if (nb == 0) nb = qr_panel_width(nmax);
  if (nb == 16 && nmax <= 512) return launch_form_Q_blocked_nb<16, 4>(s, chains, nchains, nmax, A, Q);
  if (nb != 8) return hipErrorInvalidValue;
  if (nchains >= kWideColChains) {
    const int cb = mfma_cols(nmax);
    if (cb) return launch_mfma_classes(k_form_Q_mfma<16>, k_form_Q_mfma<8>, s, nchains, nmax, chains, A, Q);
  }
  return launch_rows(k_form_Q_rows<1>, k_form_Q_rows<2>, k_form_Q_rows<3>, k_form_Q_rows<4>, s, chains, nchains, nmax, A,
                     Q);
}

hipError_t launch_qr_solve(hipStream_t s, const ChainDesc* chains, int nchains, int nmax, MatRef A, MatRef B, int nb) {
  if (nmax > kQrMaxN || nmax < 16) return hipErrorInvalidValue;
  if (nb == 0) nb = qr_panel_width(nmax);
  if (nb == 16 && nmax <= 512) return launch_qr_solve_nb<16, 4>(s, chains, nchains, nmax, A, B);
  if (nb != 8) return hipErrorInvalidValue;
  if (nchains >= kWideColChains) {
    const int cb = mfma_cols(nmax);
    if (cb) return launch_mfma_classes(k_qr_solve_mfma<16>, k_qr_solve_mfma<8>, s, nchains, nmax, chains, A, B);
  }
  return launch_rows(k_qr_solve_rows<1>, k_qr_solve_rows<2>, k_qr_solve_rows<3>, k_qr_solve_rows<4>, s, chains, nchains,
                     nmax, A, B);
}

}  // namespace dqmc
