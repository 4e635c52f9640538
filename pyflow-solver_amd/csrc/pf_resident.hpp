// Resident solves: the CG iterations of one cavity run inside one launch, its
// workgroups exchanging partial sums and region edges through memory.
//
// Protocol
// --------
// A cavity of at most one region per workgroup and at most one workgroup per
// CU can have all its workgroups on the GPU at once. When a solve's CG phase
// begins, its workgroups first meet (resident_enter): each adds itself to the
// launch's arrival word. If all arrive within KArgs::meet_ticks every workgroup is
// known to be running and the solve goes on in this launch; if one of them
// times out first (the GPU is shared with other work) it marks the word, all
// of them see the mark, and the launch runs one ordinary round, like a launch
// without this path. Afterwards each wait is for a workgroup that is running,
// so it ends; all are bounded by kWaitTicks nevertheless, after which the
// launch gives up and reports an error.
//
// Nothing is fenced. Values cross between workgroups only through relaxed
// device-scope atomic loads and stores, which reach past the per-XCD L2s, and
// every value that is waited for announces itself:
//   partial sums  64-bit words that hold kSent (all ones) until their writer
//                 stores the sum; workgroup 0 collects them, folds them as the
//                 next round would, runs the tail, and puts kSent back. Two
//                 buffers alternate, so a word is reset long before it is
//                 written again;
//   tail results  words of 32 bits of payload and a 32-bit sequence number,
//                 stored by workgroup 0 on kCopies lines (fewer readers per line);
//   region edges  FP64: one inbox per region side, read by that region only,
//                 which puts kSent back; two buffers alternate here too.
//                 MIXED: z = M r and p of the two rows or columns per side that
//                 a neighbour's frame needs, packed per region (stores past the
//                 L2s cost by the line: at 1024^2, cells stored in place in the
//                 grid took a round from 6.5 to 7.4 us), followed by the region's
//                 sequence number once the stores have completed; its neighbours
//                 wait for that number. Two buffers alternate.
// A sum or cell that equals kSent (a NaN) is stored as another NaN.
#pragma once

namespace pf {

constexpr unsigned long long kSent = ~0ull;
constexpr unsigned long long kOtherNan = 0x7ff8000000000000ull;
constexpr int kCopies = 8;
constexpr int kResMaxBlk = 256;           // workgroups of a resident cavity
constexpr long long kWaitTicks = 1000000000;  // 10 s
constexpr double kTinyD = 0x1p-300;
constexpr unsigned kMeetAbort = 0x10000u;

// Exchange block of a cavity, at KArgs::res + PfCav::res_off (bytes; the parts
// start on 128-byte lines). W = words per partial-sum slot, one a workgroup.
constexpr size_t kResMeet = 0;      // arrival words, one per round parity, 128 bytes apart
constexpr size_t kResBcast = 512;   // FP64: kCopies lines of 16 words
constexpr size_t kResTotal = 2048;  // MIXED: kCopies lines of 2 KCA words (256 bytes each)
constexpr size_t kResPart = 4096;   // FP64: [2][3][W] words; MIXED: [4][KCA][W]
__host__ __device__ constexpr size_t res_w(int nblk) { return ((size_t)nblk + 15) / 16 * 16; }
// FP64: inboxes [2][nblk][4 sides][64] words.
__host__ __device__ constexpr size_t res64_inbox(int nblk) { return kResPart + 2 * 3 * res_w(nblk) * 8; }
__host__ __device__ constexpr size_t res64_bytes(int nblk) { return res64_inbox(nblk) + (size_t)2 * nblk * 4 * 64 * 8; }
// MIXED: a sequence number per workgroup, 128 bytes apart.
__host__ __device__ constexpr size_t res32_flag(int nblk) { return kResPart + 4 * KCA * res_w(nblk) * 8; }
// MIXED: edges [2][nblk][4 sides][128] words of (z, p): the two columns (row by
// row) or rows a neighbour's frame needs from that side.
__host__ __device__ constexpr size_t res32_edge(int nblk) { return res32_flag(nblk) + (size_t)nblk * 128; }
__host__ __device__ constexpr size_t res32_bytes(int nblk) { return res32_edge(nblk) + (size_t)2 * nblk * 4 * 128 * 8; }
enum { SIDE_W = 0, SIDE_E = 1, SIDE_S = 2, SIDE_N = 3 };

constexpr int kResPitch = TX + 3;  // LDS pitch of the FP64 direction: 64 columns, a ring, odd
__host__ __device__ constexpr int res64_lds_doubles(int m) { return (TY * m + 2) * kResPitch; }

__device__ inline void dev_store(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned long long dev_load(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void dev_store_f64(unsigned long long* p, double v) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  dev_store(p, u == kSent ? kOtherNan : u);
}
// Every memory operation of this wave has completed.
__device__ inline void drain_vmem() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Words a workgroup shares during a resident solve.
struct ResShared {
  double val[2];          // FP64: alpha, beta
  float coef[4];          // MIXED: alpha_k, beta_k, alpha_k+1, beta_k+1
  double tot[KCA];        // MIXED: totals of the round
  double wtot[KCA][NWAVE + 2];  // MIXED: wave totals (rows 144 bytes apart: 14 lanes read a row each)
  double wsum[3][NWAVE];  // wave totals: P, and the two of Q
  unsigned seq0;        // sequence number of the last broadcast before this launch
  unsigned nbseq;  // MIXED: round whose edges all neighbours have published
  int go, dead, inc;
  int tiny[2];  // some d of the region or its ring is a tiny number, by iteration parity
};

// Whether this launch's workgroups are all running (see above). Every thread
// of every workgroup of the cavity calls it once per launch at most.
__device__ inline bool resident_enter(const KArgs& KA, const PfCav& C, int b, ResShared* sh) {
  if (KA.res == nullptr) return false;
  const int nblk = C.nblk;
  if (tid_flat() == 0) {
    sh->dead = 0;
    sh->go = 1;
    sh->seq0 = 0;
    sh->tiny[0] = sh->tiny[1] = 0;
    if (nblk > 1) {
      char* const res = KA.res + C.res_off;
      unsigned* meet = (unsigned*)(res + kResMeet + 128 * KA.parity);
      // The last sequence number: FP64 counts broadcasts, MIXED rounds (its flag).
      const unsigned long long* last = (const unsigned long long*)(
          C.prec == PF_PREC_MIXED ? res + res32_flag(nblk) + 128 * b : res + kResBcast + 128 * (b & (kCopies - 1)));
      const unsigned long long w = dev_load(last);
      sh->seq0 = C.prec == PF_PREC_MIXED ? (unsigned)w : (unsigned)(w >> 32);
      sh->nbseq = sh->seq0;
      drain_vmem();  // read before arriving: workgroup 0 broadcasts only after every arrival
      const long long t0 = wall_clock64();
      unsigned cur = __hip_atomic_fetch_add(meet, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
      while (true) {
        if (cur & kMeetAbort) {
          sh->go = 0;
          break;
        }
        if (cur == (unsigned)nblk) break;
        if (wall_clock64() - t0 > KA.meet_ticks) {
          unsigned want = cur | kMeetAbort;
          if (__hip_atomic_compare_exchange_strong(meet, &cur, want, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT)) {
            sh->go = 0;
            break;
          }
          continue;  // cur holds the word that won
        }
        __builtin_amdgcn_s_sleep(1);
        cur = __hip_atomic_load(meet, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  __syncthreads();
  return sh->go != 0;
}
// The previous launch's arrival word, for the launch after this one.
__device__ inline void resident_clear_meet(const KArgs& KA, const PfCav& C) {
  if (KA.res != nullptr)
    __hip_atomic_store((unsigned*)(KA.res + C.res_off + kResMeet + 128 * (KA.parity ^ 1)), 0u, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Word `lane` (0 .. nw-1) of the broadcast with sequence number `seq`, polled
// by one whole wave. False after kWaitTicks.
__device__ inline bool bcast_wait(const unsigned long long* line, int lane, int nw, unsigned seq, unsigned& payload) {
  const long long t0 = wall_clock64();
  while (true) {
    const unsigned long long w = (lane < nw) ? dev_load(line + lane) : ((unsigned long long)seq << 32);
    payload = (unsigned)w;
    if (!__any((unsigned)(w >> 32) != seq)) return true;
    if (wall_clock64() - t0 > kWaitTicks) return false;
  }
}
// The values of kSent-marked words q = lane + 64 t (t < 4, q < n), polled by one
// whole wave. False after kWaitTicks.
__device__ inline bool words_poll(const unsigned long long* w, int lane, int n, double (&v)[4]) {
  const long long t0 = wall_clock64();
  unsigned long long x[4];
  while (true) {
    bool miss = false;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int q = lane + 64 * t;
      x[t] = (q < n) ? dev_load(w + q) : 0ull;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) miss |= x[t] == kSent;
    if (!__any(miss)) break;
    if (wall_clock64() - t0 > kWaitTicks) return false;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) v[t] = __longlong_as_double((long long)x[t]);
  return true;
}
__device__ inline void words_reset(unsigned long long* w, int lane, int n) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int q = lane + 64 * t;
    if (q < n) dev_store(w + q, kSent);
  }
}
// The fold of a round's preamble: per lane in increasing workgroup order, then
// the DPP tree; the total is broadcast from lane 63.
__device__ inline double fold_words(int lane, int n, const double (&v)[4]) {
  double a = 0.0;
#pragma unroll
  for (int t = 0; t < 4; ++t)
    if (lane + 64 * t < n) a = a + v[t];
  a = wave_reduce<false>(a);
  const long long bits = __double_as_longlong(a);
  const int lo = __builtin_amdgcn_readlane((int)(bits & 0xffffffffll), 63);
  const int hi = __builtin_amdgcn_readlane((int)(bits >> 32), 63);
  return __longlong_as_double((long long)(unsigned)lo | ((long long)hi << 32));
}
// The sum of the wave totals in wave order (block_partials_k's fold).
__device__ inline double fold_waves(const double* w) {
  double t = w[0];
#pragma unroll
  for (int k = 1; k < NWAVE; ++k) t = t + w[k];
  return t;
}

// The CG iterations of an FP64 solve (phases P and Q of chunk_p / chunk_q and
// their tails), from a P phase to the end of the solve or KArgs::res_iters of them.
// A thread keeps x, r, d and q = A d of its M cells in registers; d is also in
// LDS with a one-cell ring, where the stencil reads it. A region's ring of r is
// received from its neighbours after every Q, and the ring's d is formed from
// it by the owner's expression, so it carries the owner's bits. Cell
// expressions, per-thread sums, block reduction, fold and tails are those of
// the rounds, in their order: the results are the bits of one launch per
// phase. What bounds it is the chain of an iteration: two sums over all
// workgroups (about 2 us each from the first store to the last reader; one
// launch per phase spends 2.5 us between kernels and as much again on the
// state, the partials and the vectors), the stencil with its six divisions, and
// four barriers. Per iteration, one launch per phase -> resident: 5.4 -> 3.8 us
// at 64^2 (one workgroup, against local_cg), 26 -> 9.0 us at 130x97,
// 23.2 -> 9.6 us at 512^2, 27.3 -> 10.1 us at 1000x700 (176 workgroups). The
// state is left as after a Q round's tail. A NaN residual leaves
// the loop (such a solve goes on one phase per launch, where a host that looks
// for NaN sees it). One workgroup: no exchange at all, every thread forms the
// tails' scalars from the wave totals.
template <int M>
__device__ __attribute__((always_inline)) inline void resident_cg64(const KArgs& KA, const PfCav& C, PfScal& st,
                                                                    ResShared& sh, double* __restrict__ lD, int b) {
  constexpr int P = kResPitch;
  const int nx = C.nx, ny = C.ny, nblk = C.nblk, tiles_x = C.tiles_x;
  const int li = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);  // = the row within a tile
  const int rx = b % tiles_x, ry = b / tiles_x;
  const int i0 = rx * TX, j0 = ry * TY * M;
  const int i = i0 + li;
  const bool multi = nblk > 1;
  const bool full = (i0 + TX <= nx) && (j0 + TY * M <= ny);
  const int op = C.op;
  const DivBy dx{C.dx, C.rdx}, dy{C.dy, C.rdy};
  const bool fast = C.fastdiv != 0;
  const double sign = (op == 0) ? -1.0 : 1.0;
  const int maxiter = C.maxiter;
  const double atol = st.inner_atol;
  double* X = (double*)C.x;
  double* R = (double*)C.r;
  double* const D0 = (double*)C.d0;
  double* const D1 = (double*)C.d1;
  int it = st.it, it_total = st.it_total;
  double rho = st.rho, beta = st.beta;

  // LDS word of cell (16 m + wave, li) and of its neighbours; a missing
  // neighbour is the cell itself, whose difference is +0 as the operator has it.
  const int c0 = (wave + 1) * P + li + 1;
  const int oE = c0 + ((i + 1 < nx) ? 1 : 0), oW = c0 - ((i > 0) ? 1 : 0);
  int oN[M], oS[M];
  double xv[M], rv[M], dv[M], qv[M], wv[M];
  bool in[M];
  unsigned idm = 0;  // identity rows among the thread's cells
  {
    const double* Dold = (it & 1) ? D0 : D1;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int j = j0 + TY * m + wave;
      in[m] = (i < nx) && (j < ny);
      const size_t k = in[m] ? (size_t)j * nx + i : 0;
      const double xx = X[k], rr = R[k], dd = Dold[k];
      xv[m] = in[m] ? xx : 0.0;
      rv[m] = in[m] ? rr : 0.0;
      dv[m] = in[m] ? dd : 0.0;
      wv[m] = jacobi_minv(C.jacobi, C.invd, nx, ny, j, i);
      const int o = c0 + TY * m * P;
      oN[m] = o + ((j + 1 < ny) ? P : 0);
      oS[m] = o - ((j > 0) ? P : 0);
      const bool id = (op == 0) ? (j == 0 && i == 0) : (j == 0 || j == ny - 1 || i == 0 || i == nx - 1);
      if (id && in[m]) idm |= 1u << m;
    }
  }
  const bool any_id = __any(idm != 0);
  // Ring: wave 4 + side holds that side's cells, one per lane.
  const int side = wave - 4;
  bool ring = false;
  double rr = 0.0, rd = 0.0, rw = 0.0;
  int ro = 0;
  char* const res = KA.res + C.res_off;
  const int W = (int)res_w(nblk);
  unsigned long long* inbox = (unsigned long long*)(res + res64_inbox(nblk));
  unsigned long long* mine = inbox;
  if (multi && side >= 0 && side < 4) {
    int gi, gj, row, col;
    if (side < 2) {
      gi = side == SIDE_W ? i0 - 1 : i0 + TX;
      gj = j0 + li;
      row = li + 1;
      col = side == SIDE_W ? 0 : TX + 1;
      ring = li < TY * M;
    } else {
      gi = i0 + li;
      gj = side == SIDE_S ? j0 - 1 : j0 + TY * M;
      row = side == SIDE_S ? 0 : TY * M + 1;
      col = li + 1;
      ring = true;
    }
    ring = ring && gi >= 0 && gi < nx && gj >= 0 && gj < ny;
    ro = ring ? row * P + col : 0;
    const size_t k = ring ? (size_t)gj * nx + gi : 0;
    const double* Dold = (it & 1) ? D0 : D1;
    rr = R[k];
    rd = Dold[k];
    rw = jacobi_minv(C.jacobi, C.invd, nx, ny, gj, gi);
    mine = inbox + ((size_t)b * 4 + side) * 64 + li;
  }
  const size_t inbuf = (size_t)nblk * 4 * 64;  // words per inbox buffer
  // Inboxes this thread's edge cells go to: columns (lanes 0 and 63), rows.
  const bool sendW = multi && li == 0 && rx > 0, sendE = multi && li == TX - 1 && i0 + TX < nx;
  const bool sendS = multi && wave == 0 && j0 > 0, sendN = multi && wave == TY - 1 && j0 + TY * M < ny;
  unsigned long long* const toCol =
      inbox + ((size_t)(sendW ? b - 1 : sendE ? b + 1 : 0) * 4 + (sendW ? SIDE_E : SIDE_W)) * 64 + wave;
  unsigned long long* const toS = inbox + ((size_t)(sendS ? b - tiles_x : 0) * 4 + SIDE_N) * 64 + li;
  unsigned long long* const toN = inbox + ((size_t)(sendN ? b + tiles_x : 0) * 4 + SIDE_S) * 64 + li;
  unsigned long long* const part = (unsigned long long*)(res + kResPart);
  unsigned long long* const bcast = (unsigned long long*)(res + kResBcast);
  unsigned long long* const line = bcast + 16 * (b & (kCopies - 1));
  unsigned seq = sh.seq0;
  double pq = 0.0, alpha = 0.0, rho_prev = rho, rnorm2 = st.rnorm2;
  bool dead = false;
  int n = 0;
  while (true) {
    unsigned long long* const pb = part + (n & 1) * 3 * W;
    // P: d = M r (first iteration) or d beta + M r, in registers and LDS.
    const bool first = (it == 0);
    if (tid_flat() == 0) sh.tiny[(n + 1) & 1] = 0;
    bool tiny = false;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const double z = wv[m] * rv[m];
      double d = first ? z : dv[m] * beta + z;
      if (!full) d = in[m] ? d : 0.0;
      dv[m] = d;
      lD[c0 + TY * m * P] = d;
      tiny = tiny || (fabs(d) < kTinyD && d != 0.0);
    }
    if (multi && side >= 0 && side < 4) {
      if (n > 0) {
        unsigned long long* const w = mine + ((n - 1) & 1) * inbuf;
        const long long t0 = wall_clock64();
        unsigned long long x;
        while (true) {
          x = ring ? dev_load(w) : 0ull;
          if (!__any(x == kSent)) break;
          if (wall_clock64() - t0 > kWaitTicks) {
            if (li == 0) sh.dead = 1;
            break;
          }
        }
        if (ring) dev_store(w, kSent);
        rr = __longlong_as_double((long long)x);
      }
      const double z = rw * rr;
      rd = first ? z : rd * beta + z;
      if (ring) lD[ro] = rd;
      tiny = tiny || (ring && fabs(rd) < kTinyD && rd != 0.0);
    }
    if (__any(tiny) && li == 0) sh.tiny[n & 1] = 1;
    __syncthreads();
    // q = A d. Differences of the region's d are zero or at least 2^-352 in
    // magnitude where no d is a tiny number, and so are what div_fast divides
    // after them; a numerator above its range gives a q that is not finite. A
    // region with a tiny d, or a thread with such a q, divides.
    bool slow = !fast || sh.tiny[n & 1] != 0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int o = TY * m * P;
      const double c = dv[m];
      const double tx = div_fast(lD[oE + o] - c, dx) - div_fast(c - lD[oW + o], dx);
      const double ty = div_fast(lD[oN[m]] - c, dy) - div_fast(c - lD[oS[m]], dy);
      qv[m] = ((0.0 + div_fast(tx, dx)) + div_fast(ty, dy)) * sign;
      slow = slow || !(fabs(qv[m]) < 0x1p900);
    }
    if (__any(slow)) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int o = TY * m * P;
        const double q = lap_coherent5<double>(dv[m], lD[oE + o], lD[oW + o], lD[oN[m]], lD[oS[m]], nx, ny,
                                               j0 + TY * m + wave, i, dx.b, dy.b) * sign;
        qv[m] = slow ? q : qv[m];
      }
    }
    if (any_id) {
#pragma unroll
      for (int m = 0; m < M; ++m)
        if ((idm >> m) & 1u) qv[m] = dv[m];
    }
    double s0 = 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (!full) qv[m] = in[m] ? qv[m] : 0.0;
      s0 += dv[m] * qv[m];
    }
    s0 = wave_reduce<false>(s0);
    if (li == 63) sh.wsum[0][wave] = s0;
    __syncthreads();
    if (!multi) {
      pq = 0.0 + fold_waves(sh.wsum[0]);
      alpha = rho / pq;
    } else {
      if (wave == 0) {
        const double t = fold_waves(sh.wsum[0]);
        if (li == 0) dev_store_f64(pb + b, t);
        bool ok = true;
        if (b == 0) {
          double v[4];
          ok = words_poll(pb, li, nblk, v);
          words_reset(pb, li, nblk);
          pq = fold_words(li, nblk, v);
          alpha = rho / pq;
          const long long u = __double_as_longlong(alpha);
          const unsigned pay = (li & 1) ? (unsigned)(u >> 32) : (unsigned)u;
          drain_vmem();
          if (li < 2 * kCopies) dev_store(bcast + 16 * (li >> 1) + (li & 1), pay | ((unsigned long long)(seq + 1) << 32));
        } else {
          unsigned pay;
          ok = bcast_wait(line, li, 2, seq + 1, pay);
          const unsigned lo = __builtin_amdgcn_readlane(pay, 0), hi = __builtin_amdgcn_readlane(pay, 1);
          alpha = __longlong_as_double((long long)((unsigned long long)lo | ((unsigned long long)hi << 32)));
        }
        if (li == 0) {
          sh.val[0] = alpha;
          if (!ok) sh.dead = 1;
        }
      }
      seq += 1;
      __syncthreads();
      alpha = sh.val[0];
      if (sh.dead) {
        dead = true;
        break;
      }
    }
    // Q: x += alpha d, r -= alpha q, partials r.(M r) and r.r; the region's
    // edges of r go to the neighbours' inboxes.
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      xv[m] = xv[m] + alpha * dv[m];
      double r = rv[m] - alpha * qv[m];
      if (!full) r = in[m] ? r : 0.0;
      rv[m] = r;
      const double z = wv[m] * r;
      s1 += r * z;
      s2 += r * r;
    }
    if (multi) {
      const size_t ob = (size_t)(n & 1) * inbuf;
      if (sendW || sendE) {
#pragma unroll
        for (int m = 0; m < M; ++m)
          if (in[m]) dev_store_f64(toCol + ob + TY * m, rv[m]);
      }
      if (sendS && in[0]) dev_store_f64(toS + ob, rv[0]);
      if (sendN && in[M - 1]) dev_store_f64(toN + ob, rv[M - 1]);
    }
    s1 = wave_reduce<false>(s1);
    s2 = wave_reduce<false>(s2);
    if (li == 63) {
      sh.wsum[1][wave] = s1;
      sh.wsum[2][wave] = s2;
    }
    __syncthreads();
    bool more = false;
    n += 1;
    it += 1;
    it_total += 1;
    if (!multi) {
      rho_prev = rho;
      rho = 0.0 + fold_waves(sh.wsum[1]);
      rnorm2 = 0.0 + fold_waves(sh.wsum[2]);
      beta = rho / rho_prev;
      more = it_total < maxiter && !(sqrt(rnorm2) < atol) && !isnan(rnorm2) && n < KA.res_iters;
    } else {
      if (wave == 0) {
        const double t1 = fold_waves(sh.wsum[1]), t2 = fold_waves(sh.wsum[2]);
        if (li < 2) dev_store_f64(pb + (1 + li) * W + b, li ? t2 : t1);
        bool ok = true;
        if (b == 0) {
          double v[4], w[4];
          ok = words_poll(pb + W, li, nblk, v);
          ok = words_poll(pb + 2 * W, li, nblk, w) && ok;
          words_reset(pb + W, li, nblk);
          words_reset(pb + 2 * W, li, nblk);
          rho_prev = rho;
          rho = fold_words(li, nblk, v);
          rnorm2 = fold_words(li, nblk, w);
          beta = rho / rho_prev;
          more = it_total < maxiter && !(sqrt(rnorm2) < atol) && !isnan(rnorm2) && n < KA.res_iters;
          const long long u = __double_as_longlong(beta);
          const int wd = li & 3;
          const unsigned pay = wd == 0 ? (unsigned)u : wd == 1 ? (unsigned)(u >> 32) : (more ? 1u : 0u);
          drain_vmem();
          if (li < 4 * kCopies && wd < 3)
            dev_store(bcast + 16 * (li >> 2) + wd, pay | ((unsigned long long)(seq + 1) << 32));
        } else {
          unsigned pay;
          ok = bcast_wait(line, li, 3, seq + 1, pay);
          const unsigned lo = __builtin_amdgcn_readlane(pay, 0), hi = __builtin_amdgcn_readlane(pay, 1);
          beta = __longlong_as_double((long long)((unsigned long long)lo | ((unsigned long long)hi << 32)));
          more = __builtin_amdgcn_readlane(pay, 2) != 0;
        }
        if (li == 0) {
          sh.val[1] = beta;
          sh.go = more ? 1 : 0;
          if (!ok) sh.dead = 1;
        }
      }
      seq += 1;
      __syncthreads();
      beta = sh.val[1];
      more = sh.go != 0;
      if (sh.dead) {
        dead = true;
        break;
      }
    }
    if (!more) break;
  }
  if (dead) {
    if (tid_flat() == 0) __hip_atomic_store(KA.active + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  // Leave the vectors and the state as a Q round and its tail leave them.
  double* Dn = ((it - 1) & 1) ? D1 : D0;  // the last P's direction array
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (in[m]) {
      const size_t k = (size_t)(j0 + TY * m + wave) * nx + i;
      X[k] = xv[m];
      R[k] = rv[m];
      Dn[k] = dv[m];
    }
  }
  if (multi && side >= 0 && side < 4) {  // the last Q's edges, which no P reads
    unsigned long long* const w = mine + ((n - 1) & 1) * inbuf;
    const long long t0 = wall_clock64();
    while (true) {
      const unsigned long long x = ring ? dev_load(w) : 0ull;
      if (!__any(x == kSent) || wall_clock64() - t0 > kWaitTicks) break;
    }
    if (ring) dev_store(w, kSent);
  }
  if (b == 0 && tid_flat() == 0) {
    st.it_run += it_total - st.it_total;
    st.it = it;
    st.it_total = it_total;
    st.pq = pq;
    st.alpha = alpha;
    st.rho_prev = rho_prev;
    st.rho = rho;
    st.rnorm2 = rnorm2;
    st.beta = beta;
    st.pending = PH_IDLE;
    cg_next(C, st);
  }
}

// LDS of resident_ca: p, z = M r and M A p on a region with its 4-cell frame,
// and x of its cells.
__host__ __device__ constexpr int res32_lds_floats(int m) { return 3 * (TY * m + 8) * HQ + m * NTH; }
// Up to this many workgroups, each collects all sums itself.
constexpr int kAllToAll = 16;

// The two-iteration PCG rounds of an inner solve of a MIXED cavity (region_ca
// and tail_ca, FP32 iterate), from a round that runs iterations to the round
// that ends the inner solve or KArgs::res_iters rounds. A thread keeps r, p, x of its M
// cells, and with them a = A p, c = A M a and e = A z: the round forms them of
// the new basis for its Gram sums, and the next round needs the same values
// again, so it evaluates three stencils per cell instead of six. p, z and M a
// lie in LDS with the frame. Of the frame, a region computes distances 1 and 2
// itself (r, p and a by their owner's expressions) and receives distances 3 and
// 4 from its neighbours after every round. All that does not depend on the new
// step lengths (receiving the frame; a at distances 2 and 3; c and e at
// distances 1 and 2) runs while the sums are under way. Cell expressions, sums,
// reduction, fold and tail are those of region_ca's rounds in their order, so the
// results are the same bits. A missing neighbour at the domain's edge is read
// as the cell itself (its difference is +0, as region_ca's ghost copies make it).
template <int M>
__device__ __attribute__((always_inline)) inline void resident_ca(const KArgs& KA, const PfCav& C, PfScal& st,
                                                                  ResShared& sh, float* __restrict__ lds, int b) {
  constexpr int RH = TY * M, NR = RH + 8, TP = TY * HQ;
  constexpr int F1 = ca_frame_cells(RH, 1), F2 = ca_frame_cells(RH, 2), F3 = ca_frame_cells(RH, 3);
  constexpr int F4 = ca_frame_cells(RH, 4);
  static_assert(F3 <= NTH && F4 <= NTH + 64, "a frame cell per thread, and one more in wave 0");
  static_assert(NR * HQ < (1 << 16), "LDS words fit 16 bits");
  float* __restrict__ lP = lds;
  float* __restrict__ lZ = lds + NR * HQ;
  float* __restrict__ lMA = lds + 2 * NR * HQ;
  float* __restrict__ lX = lds + 3 * NR * HQ + threadIdx.y * TX + threadIdx.x;  // cell m at lX[m * NTH]
  const int nx = C.nx, ny = C.ny, nblk = C.nblk, tiles_x = C.tiles_x;
  const int li = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int tid = wave * TX + li;
  const int rx = b % tiles_x, ry = b / tiles_x;
  const int i0 = rx * TX, j0 = ry * RH;
  const int i = i0 + li;
  const bool pinned = (C.op == 0);
  const float scx = pinned ? -C.cxf : C.cxf, scy = pinned ? -C.cyf : C.cyf;
  const int rows = min(RH, ny - j0);  // rows of the region inside the domain
  auto minv = [&](int j, int ii) -> float {
    if (!C.jacobi) return 1.0f;
    return (ii == 0 || ii == nx - 1 || j == 0 || j == ny - 1) ? 1.0f : C.invdf;
  };
  auto ident = [&](int j, int ii) -> bool {
    return pinned ? (j == 0 && ii == 0) : (j == 0 || j == ny - 1 || ii == 0 || ii == nx - 1);
  };
  auto lap = [&](const float* L, float c, int oe, int ow, int on, int os) -> float {
    return __fmul_rn((L[oe] - c) - (c - L[ow]), scx) + __fmul_rn((L[on] - c) - (c - L[os]), scy);
  };
  char* const res = KA.res + C.res_off;
  const int par = KA.parity ^ st.flip;  // of the r and p buffers
  const int W = (int)res_w(nblk);

  // Own cells. East and west neighbours by offset (the cell itself where there
  // is none); across the domain's lower and upper edge the wave that holds the
  // edge row keeps a copy of it in the LDS row beyond (egS, egN: bit m).
  const int o0 = (wave + 4) * HQ + li + 4;
  const int oE = o0 + ((i + 1 < nx) ? 1 : 0), oW = o0 - ((i > 0) ? 1 : 0);
  float ro[M], po[M], ao[M], cv[M], ev[M], mo[M];
  unsigned idm = 0;              // identity rows (bit m)
  unsigned inr = 0, egN = 0;     // wave-uniform: row m is in the domain; is its last row
  const unsigned egS = (wave == 0 && j0 == 0) ? 1u : 0u;
  {
    const float* __restrict__ R = mixed_r(C, par);
    const float* __restrict__ Pold = mixed_p(C, par ^ 1);
    const float* __restrict__ X = (const float*)C.x;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int row = TY * m + wave, j = j0 + row;
      const bool in = (i < nx) && (j < ny);
      const unsigned k = in ? (unsigned)(j * nx + i) : 0u;
      ro[m] = R[k];
      po[m] = Pold[k];
      lX[m * NTH] = X[k];
      mo[m] = minv(j, i);
      if (j < ny) inr |= 1u << m;
      if (j == ny - 1) egN |= 1u << m;
      if (in && ident(j, i)) idm |= 1u << m;
    }
  }
  const bool full = (i0 + TX <= nx) && rows == RH;
  const bool edges = (egS | egN) != 0;
  const bool any_id = __any(idm != 0);
  auto own_put = [&](float* L, int m, float v) {
    if ((inr >> m) & 1u) L[o0 + m * TP] = v;
    if (edges) {
      if ((egN >> m) & 1u) L[o0 + m * TP + HQ] = v;
      if ((egS >> m) & 1u) L[o0 + m * TP - HQ] = v;
    }
  };
  // Frame cells: q0 per thread, counted down so that wave 0, which also waits
  // for the totals, has the outermost; q1 in wave 0 where the frame has more
  // than NTH cells. f: LDS word; bits 16-19 the neighbours it has (E, W, N, S),
  // 20 identity row, 21-23 within distance 1, 2, 3, 24 received (3 or 4), 25
  // Jacobi weight 1. Its p is read back from LDS.
  const int q0 = NTH - 1 - tid;
  unsigned f = 0, fk = 0, g = 0, gk = 0;  // fk, gk: byte offsets of received cells among the edges
  // Byte offset of the cell at (row, col) of the frame, distance 3 or 4, among
  // the edges: its region, and which of that region's sides has it.
  auto edge_of = [&](int row, int col) -> unsigned {
    const int dy = row < 4 ? row - 4 : (row >= RH + 4 ? row - RH - 3 : 0);  // signed distance from the region
    const int dx = col < 4 ? col - 4 : (col >= TX + 4 ? col - TX - 3 : 0);
    const int reg = b + (dx > 0 ? 1 : dx < 0 ? -1 : 0) + (dy > 0 ? tiles_x : dy < 0 ? -tiles_x : 0);
    int side, w;
    if (dx <= -3 || dx >= 3) {  // its east columns TX-4, TX-3 or its west columns 2, 3
      side = dx < 0 ? SIDE_E : SIDE_W;
      const int r = dy == 0 ? row - 4 : dy < 0 ? RH + dy : dy - 1;
      w = 2 * r + (dx < 0 ? dx + 4 : dx - 3);
    } else {
      side = dy < 0 ? SIDE_N : SIDE_S;
      const int q = dx == 0 ? col - 4 : dx < 0 ? TX + dx : dx - 1;
      w = (dy < 0 ? dy + 4 : dy - 3) * TX + q;
    }
    return 8u * (unsigned)((reg * 4 + side) * 128 + w);
  };
  float fr = 0.f, fa = 0.f, fc = 0.f, fe = 0.f;
  auto weight = [&]() -> float { return (f & (1u << 25)) ? 1.0f : C.invdf; };
  {
    const float* __restrict__ R = mixed_r(C, par);
    const float* __restrict__ Pold = mixed_p(C, par ^ 1);
    int row = 0, col = 0;
    if (q0 < F4) ca_frame_cell(RH, q0, row, col);
    int gj = j0 + row - 4, gi = i0 + col - 4;
    if (q0 < F4 && gi >= 0 && gi < nx && gj >= 0 && gj < ny) {
      f = (unsigned)(row * HQ + col);
      if (gi + 1 < nx) f |= 1u << 16;
      if (gi > 0) f |= 1u << 17;
      if (gj + 1 < ny) f |= 1u << 18;
      if (gj > 0) f |= 1u << 19;
      if (ident(gj, gi)) f |= 1u << 20;
      if (q0 < F1) f |= 1u << 21;
      if (q0 < F2) f |= 1u << 22;
      if (q0 < F3) f |= 1u << 23;
      if (q0 >= F2) f |= 1u << 24;
      if (minv(gj, gi) == 1.0f) f |= 1u << 25;
      const unsigned k = (unsigned)(gj * nx + gi);
      if (q0 >= F2) fk = edge_of(row, col);
      fr = R[k];
      lP[f & 0xffffu] = Pold[k];
      lZ[f & 0xffffu] = weight() * fr;
    }
    if (F4 > NTH && NTH + tid < F4) {
      ca_frame_cell(RH, NTH + tid, row, col);
      gj = j0 + row - 4;
      gi = i0 + col - 4;
      if (gi >= 0 && gi < nx && gj >= 0 && gj < ny) {
        g = (unsigned)(row * HQ + col) | (1u << 24);
        const unsigned k = (unsigned)(gj * nx + gi);
        gk = edge_of(row, col);
        lP[g & 0xffffu] = Pold[k];
        lZ[g & 0xffffu] = minv(gj, gi) * R[k];
      }
    }
  }
  // The word of the edges this thread publishes after every round, if any (e:
  // LDS word of its cell, bit 24 set): 128 threads per side that has a neighbour.
  unsigned e = 0;
  if (tid < 512) {
    const int side = tid >> 7, w = tid & 127;
    const int row = side < 2 ? w >> 1 : (side == SIDE_S ? 2 : RH - 4) + (w >> 6);
    const int col = side < 2 ? (side == SIDE_W ? 2 : TX - 4) + (w & 1) : w & 63;
    const bool to = side == SIDE_W ? rx > 0 : side == SIDE_E ? i0 + TX < nx : side == SIDE_S ? j0 > 0 : j0 + RH < ny;
    if (to && row < rows && i0 + col < nx) e = (unsigned)((row + 4) * HQ + col + 4) | (1u << 24);
  }
  // The neighbour whose sequence number lane 0..7 of wave 15 watches, else the
  // region itself.
  int watch = b;
  if (li < 8) {
    const int t = li < 4 ? li : li + 1;  // 3 x 3 without the centre
    const int nxr = rx + t % 3 - 1, nyr = ry + t / 3 - 1;
    if (nxr >= 0 && nxr < tiles_x && nyr >= 0 && nyr * RH < ny) watch = nyr * tiles_x + nxr;
  }
  const unsigned seq0 = sh.seq0;
  // Which slots this wave collects: every workgroup all of them (wave k slot k),
  // or workgroup b the slots k = b mod nown, in waves 8 and up.
  const bool multi = nblk > 1, all = nblk <= kAllToAll;
  const int nown = min(nblk, KCA);
  const int slot = all ? wave : (wave >= 8 && b < nown ? b + (wave - 8) * nown : KCA);
  int it_total = st.it_total, inc = st.ca_inc;

  // The stencils of the first basis.
#pragma unroll
  for (int m = 0; m < M; ++m) {
    own_put(lP, m, po[m]);
    own_put(lZ, m, mo[m] * ro[m]);
  }
  __syncthreads();
  auto own_a = [&]() {  // a = A p, M a into LDS
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int d = m * TP;
      ao[m] = lap(lP, po[m], oE + d, oW + d, o0 + d + HQ, o0 + d - HQ);
      if (any_id) ao[m] = ((idm >> m) & 1u) ? po[m] : ao[m];
      own_put(lMA, m, mo[m] * ao[m]);
    }
  };
  auto own_ce = [&](int m) {  // c = A M a, e = A z
    const int d = m * TP;
    const float ma = mo[m] * ao[m], z = mo[m] * ro[m];
    cv[m] = lap(lMA, ma, oE + d, oW + d, o0 + d + HQ, o0 + d - HQ);
    ev[m] = lap(lZ, z, oE + d, oW + d, o0 + d + HQ, o0 + d - HQ);
    if (any_id) {
      cv[m] = ((idm >> m) & 1u) ? ma : cv[m];
      ev[m] = ((idm >> m) & 1u) ? z : ev[m];
    }
  };
  auto frame_lap = [&](const float* L, float c) -> float {
    const int o = f & 0xffffu;
    const float v = lap(L, c, o + ((f >> 16) & 1u), o - ((f >> 17) & 1u), o + ((f >> 18) & 1u) * HQ,
                        o - ((f >> 19) & 1u) * HQ);
    return (f & (1u << 20)) ? c : v;
  };
  auto frame_a = [&]() {
    fa = frame_lap(lP, lP[f & 0xffffu]);
    lMA[f & 0xffffu] = weight() * fa;
  };
  auto frame_ce = [&]() {
    fc = frame_lap(lMA, weight() * fa);
    fe = frame_lap(lZ, weight() * fr);
  };
  own_a();
  if (f & (1u << 23)) frame_a();
  __syncthreads();
#pragma unroll
  for (int m = 0; m < M; ++m) own_ce(m);
  if (f & (1u << 22)) frame_ce();
  float a0 = (float)st.ca0, b0 = (float)st.cb0, a1 = (float)st.ca1, b1 = (float)st.cb1;
  __syncthreads();
  bool dead = false;
  int n = 0;
  while (true) {
    const unsigned seq = seq0 + 1 + (unsigned)n;
    // What derives from these is formed where it is used: hoisted out of the
    // loop it would be spilled, and a reload waits for the stores before it.
    int lv = li;
    asm volatile("" : "+v"(f), "+v"(fk), "+v"(g), "+v"(gk), "+v"(e), "+v"(watch), "+v"(lv));
    char* const xb = res + res32_edge(nblk) + ((n & 1) ? (size_t)nblk * 4096 : 0);
    // The two steps (ca_steps).
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float z = mo[m] * ro[m], ma = mo[m] * ao[m];
      const float p1 = (z - a0 * ma) + b0 * po[m];
      const float ap1 = (ev[m] - a0 * cv[m]) + b0 * ao[m];
      lX[m * NTH] = (lX[m * NTH] + a0 * po[m]) + a1 * p1;
      ro[m] = (ro[m] - a0 * ao[m]) - a1 * ap1;
      const float z2 = mo[m] * ro[m];
      po[m] = z2 + b1 * p1;
      own_put(lP, m, po[m]);
      own_put(lZ, m, z2);
    }
    if (f & (1u << 22)) {
      const float fm = weight(), fp = lP[f & 0xffffu];
      const float z = fm * fr, ma = fm * fa;
      const float p1 = (z - a0 * ma) + b0 * fp;
      const float ap1 = (fe - a0 * fc) + b0 * fa;
      fr = (fr - a0 * fa) - a1 * ap1;
      const float z2 = fm * fr;
      lP[f & 0xffffu] = z2 + b1 * p1;
      lZ[f & 0xffffu] = z2;
    }
    __syncthreads();
    if (e) {
      const unsigned o = e & 0xffffu;
      dev_store((unsigned long long*)(xb + 8u * (unsigned)(b * 512 + wave * TX + lv)),
                (unsigned long long)__float_as_uint(lZ[o]) | ((unsigned long long)__float_as_uint(lP[o]) << 32));
    }
    own_a();
    if (f & (1u << 21)) frame_a();
    __syncthreads();
    // c, e and the Gram sums of the new basis (pass 5 of region_ca).
    double acc[NP] = {0.0, 0.0, 0.0, 0.0};
    auto gram = [&](int m) {
      const double p2 = po[m], z2 = mo[m] * ro[m], r2 = ro[m], a2 = ao[m];
      const double ma2 = mo[m] * ao[m], c2 = cv[m], mc2 = mo[m] * cv[m], e2 = ev[m], me2 = mo[m] * ev[m];
      acc[0] = __fma_rn(p2, a2, acc[0]);
      acc[1] = __fma_rn(p2, c2, acc[1]);
      acc[2] = __fma_rn(p2, e2, acc[2]);
      acc[3] = __fma_rn(a2, ma2, acc[3]);
      acc[4] = __fma_rn(a2, mc2, acc[4]);
      acc[5] = __fma_rn(a2, z2, acc[5]);
      acc[6] = __fma_rn(a2, me2, acc[6]);
      acc[7] = __fma_rn(c2, mc2, acc[7]);
      acc[8] = __fma_rn(c2, z2, acc[8]);
      acc[9] = __fma_rn(c2, me2, acc[9]);
      acc[10] = __fma_rn(r2, z2, acc[10]);
      acc[11] = __fma_rn(z2, e2, acc[11]);
      acc[12] = __fma_rn(e2, me2, acc[12]);
      acc[13] = __fma_rn(r2, r2, acc[13]);
    };
    if (full) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        own_ce(m);
        gram(m);
      }
    } else {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        own_ce(m);
        if (((inr >> m) & 1u) && i < nx) gram(m);
      }
    }
    wave_partials_ca(acc, [&](int k, double v) { sh.wtot[k][wave] = v; });
    drain_vmem();  // the published cells are in memory before the barrier, so before the flag
    __syncthreads();
    unsigned long long* const pb = (unsigned long long*)(res + kResPart) + (size_t)(seq & 3) * KCA * W;
    if (wave == 0 && lv < KCA) {
      const double t = fold_waves(sh.wtot[lv]);
      if (multi)
        dev_store_f64(pb + lv * W + b, t);
      else
        sh.tot[lv] = 0.0 + t;
    }
    if (multi) {
      if (wave == NWAVE - 1) {
        unsigned long long* const flags = (unsigned long long*)(res + res32_flag(nblk));
        if (li == 0) dev_store(flags + 16 * b, (unsigned long long)seq);
        const long long t0 = wall_clock64();
        while (true) {
          const unsigned w = li < 8 ? (unsigned)dev_load(flags + 16 * watch) : seq;
          if (!__any((int)(w - seq) < 0)) break;
          if (wall_clock64() - t0 > kWaitTicks) {
            if (li == 0) sh.dead = 1;
            break;
          }
        }
        if (li == 0) __hip_atomic_store(&sh.nbseq, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      // Waves that receive wait for that (wave 15's wait is bounded).
      if (__any(((f | g) >> 24) & 1u)) {
        while (__hip_atomic_load(&sh.nbseq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != seq)
          __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
      }
      unsigned long long fx = 0, gx = 0;
      if (f & (1u << 24)) fx = dev_load((const unsigned long long*)(xb + fk));
      if (g) gx = dev_load((const unsigned long long*)(xb + gk));
      if (slot < KCA) {
        bool ok = true;
        for (int k = slot; k < KCA; k += all ? KCA : 8 * nown) {
          double v[4];
          ok = words_poll(pb + k * W, lv, nblk, v) && ok;
          const double t = fold_words(lv, nblk, v);
          if (all) {
            if (li == 0) sh.tot[k] = t;
          } else {
            const unsigned long long u = (unsigned long long)__double_as_longlong(t);
            const unsigned pay = (lv & 1) ? (unsigned)(u >> 32) : (unsigned)u;
            unsigned long long* const total = (unsigned long long*)(res + kResTotal);
            if (lv < 2 * kCopies) dev_store(total + 32 * (lv >> 1) + 2 * k + (lv & 1), pay | ((unsigned long long)seq << 32));
            words_reset(pb + k * W, lv, nblk);
          }
        }
        if (!ok && li == 0) sh.dead = 1;
      }
      // Each workgroup puts its own words of the round before (the last one of
      // the launch before, if this is the first) back to kSent: every workgroup has
      // read them, since all have stored this round's.
      if (all && wave == 0 && lv < KCA)
        dev_store((unsigned long long*)(res + kResPart) + ((size_t)((seq + 3) & 3) * KCA + lv) * W + b, kSent);
      if (f & (1u << 24)) {
        lZ[f & 0xffffu] = __uint_as_float((unsigned)fx);
        lP[f & 0xffffu] = __uint_as_float((unsigned)(fx >> 32));
      }
      if (g) {
        lZ[g & 0xffffu] = __uint_as_float((unsigned)gx);
        lP[g & 0xffffu] = __uint_as_float((unsigned)(gx >> 32));
      }
    }
    __syncthreads();
    if ((f & (5u << 21)) == (4u << 21)) frame_a();  // distances 2 and 3
    __syncthreads();
    it_total += inc;
    if (wave == 0) {
      if (!all) {
        unsigned pay;
        const unsigned long long* const line = (const unsigned long long*)(res + kResTotal) + 32 * (b & (kCopies - 1));
        const bool ok = bcast_wait(line, lv, 2 * KCA, seq, pay);
        if (lv < 2 * KCA) ((unsigned*)sh.tot)[lv] = pay;
        if (!ok && li == 0) sh.dead = 1;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
      const CaTail r = tail_ca_steps(sh.tot, it_total, C.maxiter, st.inner_atol);
      if (li == 0) {
        sh.coef[0] = (float)r.a0;
        sh.coef[1] = (float)r.b0;
        sh.coef[2] = (float)r.a1;
        sh.coef[3] = (float)r.b1;
        sh.inc = r.n;
        sh.go = (r.next == 0 && n + 1 < KA.res_iters) ? 1 : 0;
        if (b == 0 && sh.go == 0) {
          st.it += it_total - st.it_total;
          st.it_run += it_total - st.it_total;
          st.it_total = it_total;
          tail_ca_store(C, st, sh.tot, r);
        }
      }
    }
    if (f & (1u << 22)) frame_ce();
    n += 1;
    __syncthreads();
    a0 = sh.coef[0];
    b0 = sh.coef[1];
    a1 = sh.coef[2];
    b1 = sh.coef[3];
    inc = sh.inc;
    dead = sh.dead != 0;
    if (dead || sh.go == 0) break;
  }
  if (dead) {
    if (tid == 0) __hip_atomic_store(KA.active + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  // Leave the vectors as a round of this parity leaves them.
  float* __restrict__ Rn = mixed_r(C, par ^ 1);
  float* __restrict__ Pn = mixed_p(C, par);
  float* __restrict__ X = (float*)C.x;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int j = j0 + TY * m + wave;
    if (i < nx && j < ny) {
      const unsigned k = (unsigned)(j * nx + i);
      Rn[k] = ro[m];
      Pn[k] = po[m];
      X[k] = lX[m * NTH];
    }
  }
}

}  // namespace pf
