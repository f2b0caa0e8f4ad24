// resident.h — the resident step: a whole run of a small grid in one launch.
// Included by rfxhip.hip inside its anonymous namespace.
//
// The two-pass step of a small grid is bound by its launches: 87 x 47 x 42
// cells take 9.5 us a step (two graph nodes), although their fields are 4 MB.  Here every workgroup keeps a block of the grid for the
// whole run -- fields, CPML memory and coefficients in registers, one thread
// per (y, z) column of NX cells along x, the fields' copies for the y and z
// neighbours in LDS -- and only the block's faces travel: the E of its low
// faces to the workgroups behind it before each H update, the H of its high
// faces to the ones ahead before each E update.
//
// A face value goes through a mailbox word of 64 bits, the float and a tag
// that names the half step, written and read with relaxed device-scope
// atomics: they are coherent over the 8 XCDs by themselves, and a word whose
// tag is right holds the right value, so there is no fence, no flag and no
// grid barrier (a grid barrier writes back and invalidates every L2 and took
// 42-79 us a step).  One exchange of 256-1024 words a workgroup was measured
// at 0.6-1.1 us, of 2048 words at 1.4-2.3 us.  Words are double-buffered by
// the parity of the step: a workgroup writes a word's second next value only
// after its reader has sent what it computed from the first.
//
// All workgroups must run together: there is at most one per compute unit, and
// the host lets one resident launch at a time onto a device.  Every wait is
// bounded all the same.  A workgroup that gives up leaves the loop within 32
// steps and sets `stop`, which ends the others' waits; what such a run computed is
// worth nothing, so k_res_check, the last kernel of every run, then makes
// all of its outputs NaN and tells the host.
//
// Measured (one step, two-pass -> resident): 28^3 cells 8.7 -> 2.85 us, 87 x 47 x
// 42 9.5 -> 4.6, 42^3 without CPML 7.9 -> 3.1, 113 x 97 x 80 16.5 -> 10.5, with a
// DFT plane 21.1 -> 11.9.  What is left is the two exchanges (0.9-1.5 us each) and, from
// 3000 cells a workgroup up, the arithmetic of the blocks in a corner of the
// CPML, which the others wait for.  What mattered in the loop: no global
// load outside the exchange (vector memory returns in order, so any other
// load waits for the mailbox stores before it: 0.4 us a step for a per-cell
// ch), source values staged for many steps, a barrier for LDS alone, lane
// conditions as bits of one register, and the z slabs' columns gathered in
// the last wavefronts (12.6 -> 10.7 us at 114 x 97 x 80).
//
// The arithmetic is that of h_core and e_core_co for kappa = 1, product for product: the
// fused multiply-adds are written out as the compiler forms them there, so
// the fields are the two-pass step's bit for bit.

constexpr int kResThreads = 512;    // most threads of a workgroup
constexpr int kResPS = 640;         // LDS floats of one plane of a block (with its halo)
constexpr int kResOps = 256;        // point operations a block may hold
constexpr int kResWave = 4096;      // source values staged at once (steps x operations)
constexpr int kResWords = 3;        // y/z halo words a thread fetches per exchange
constexpr int kResEdge = 192;       // most rows plus columns of a block
constexpr int kResSnaps = 32;       // DFT planes, flux monitors and NTFF faces
constexpr int kResLook = 1 << 12;   // polls between a wait's looks at whether to give up
constexpr int kResSpin = 1 << 22;   // polls before it does so by itself (seconds)

typedef unsigned long long u64;

// A plane (or plane region) whose values every step leaves in a staging ring
// [steps of a launch][ncomp][npts], for k_res_fold to add up afterwards.
struct ResSnap {
  float* out;
  int axis, index, lo1, hi1, lo2, hi2;
  int comp[4], ncomp, avg;          // avg: H averaged over the planes index-1 and index
  int n2;
  long long npts;
};

struct ResIO {
  float* f[6];                      // state, updated in place
  float* psi;                       // CPML memory of the current set (null: none)
  unsigned foff[6], fs[6];          // each face's terms in it (as TBCpml)
  const float* src_wave;            // the plan's point-operation tables
  float* probe_out;
  float* port_out;
  int n_src, n_probe, n_port;
  u64* box;                         // mailboxes [phase][parity][workgroup][words]
  unsigned* stop;                   // set by a workgroup that gave up
  int spin;                         // polls before a wait gives up
  const ResSnap* snaps;
  int n_snap;
  int ty, tz, ntx, nty, ntz;        // tile rows, columns; tiles per axis
  int n_steps;
  long long step0;
  unsigned tag0;                    // this launch's tags are tag0 + 1 .. tag0 + 2 n_steps
};

// A point operation of the block, staged in LDS in the order of its cell's
// thread and then of the plan, so that a thread's operations lie together.
struct ResOp {
  int own;          // thread * NX + plane of the cell
  int kind, comp, slot;
  float d_par;
  float loop[3];
};

template <int NX>
struct ResShared {
  float e[3][NX][kResPS];           // row r, column c at r * (tz + 1) + c; halo row ty, column tz
  float h[3][NX][kResPS];           // at (r + 1) * (tz + 1) + c + 1; halo row and column 0
  float4 xprof[NX];                 // (b, c, 1/size, 0) of an x slab's planes
  ResOp ops[kResOps];               // the block's point operations
  float w[kResWave];                // their source values of the next steps [step][operation]
  float gx[2][NX];                  // graded: the planes' inverse spacings (H, E)
  ResSnap snap[kResSnaps];
  int n_ops, bad, spin;             // bad: a wait gave up
  int wcnt[kResThreads / 64];
};

// Mailbox word at a byte offset from a (wave-uniform) base.
__device__ __forceinline__ u64 res_ld(const u64* base, unsigned off) {
  return __hip_atomic_load((const RFX_G u64*)((const RFX_G char*)base + off), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}
// Two values of a cell in neighbouring words.
__device__ __forceinline__ void res_st2(u64* base, unsigned off, float a, float b, unsigned tag) {
  RFX_G u64* const w = (RFX_G u64*)((RFX_G char*)base + off);
  __hip_atomic_store(w, ((u64)tag << 32) | __float_as_uint(a), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(w + 1, ((u64)tag << 32) | __float_as_uint(b), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}
// Words of a workgroup's mailbox: the x face, one pair per thread, then per
// plane the y face's pairs (by column) and the z face's (by row).
constexpr unsigned res_words(int nx) { return 2u * (kResThreads + (unsigned)nx * kResEdge); }

// iy * a - iz * b and the memory's recursion, as the two-pass kernels round them.
__device__ __forceinline__ float res_curl(float i1, float a, float i2, float b) {
#pragma clang fp contract(off)
  const float t = i2 * b;
  return __builtin_fmaf(i1, a, -t);
}
__device__ __forceinline__ float res_psi(float b, float psi, float c, float g) {
#pragma clang fp contract(off)
  const float t = b * psi;
  return __builtin_fmaf(c, g, t);
}
// One slab term pair of an axis: the memory m0, m1 advanced, the corrections
// in d0, d1 (kappa is 1 in every slab: the plan checks that 1/kappa - 1 = 0,
// so the correction is the memory's product alone).
struct ResSlab {
  float b, c, inv;
};
__device__ __forceinline__ void res_slab(const ResSlab& s, float co, float g0, float g1, float& m0,
                                         float& m1, float& d0, float& d1) {
#pragma clang fp contract(off)
  m0 = res_psi(s.b, m0, s.c, g0 * s.inv);
  m1 = res_psi(s.b, m1, s.c, g1 * s.inv);
  d0 = co * m0;
  d1 = co * m1;
}

template <bool GRADED, int NX>
__global__ __launch_bounds__(kResThreads) void k_resident(const KParams* __restrict__ pp,
                                                          ResIO io) {
  __shared__ ResShared<NX> sh;
  constexpr int G = NX < 4 ? NX : NX == 4 ? 4 : 2;  // cells whose neighbours are in flight together
  const int tid = (int)threadIdx.x, T = (int)blockDim.x;
  const int ty = io.ty, tz = io.tz, tyz = ty * tz, rs = tz + 1;
  const int wg = (int)blockIdx.x, n_wg = (int)gridDim.x;
  const int bz = wg % io.ntz, by = (wg / io.ntz) % io.nty, bx = wg / (io.ntz * io.nty);
  // Thread to (row, column): the columns outside the z slabs first, row by
  // row, then those inside, so that only the last wavefronts run the z slabs'
  // code (with the columns in order every wavefront has some of them).
  const int sz_lo = min(max(pp->cn[4] - bz * tz, 0), tz);
  const int sz_hi = min(max(bz * tz + tz - (pp->nz - pp->cn[5]), 0), tz - sz_lo);
  const int n_in = tz - sz_lo - sz_hi, n_sl = sz_lo + sz_hi;
  int row, col;
  if (tid < ty * n_in) {
    row = tid / n_in;
    col = sz_lo + tid - row * n_in;
  } else if (n_sl > 0) {
    const int u = tid - ty * n_in;
    row = u / n_sl;
    col = u - row * n_sl;
    if (col >= sz_lo) col += n_in;
  } else {
    row = ty;                       // past the block
    col = 0;
  }
  const int i0 = bx * NX, j = by * ty + row, k = bz * tz + col;
  const bool in_tile = tid < tyz;

  // Per-thread constants of the loop.  Everything that only the way in and
  // out needs (field pointers, slab addresses) is read from the parameter
  // block again at the end: held across the loop it would fill the scalar
  // registers and spill.
  float ex[NX], ey[NX], ez[NX], hx[NX], hy[NX], hz[NX];
  float ca[NX], cb[NX], ce[NX];
  // 4 bits per cell: E components held at zero (outer PEC faces, PEC mask,
  // cells outside the grid)
  unsigned fl = 0u;
  float px[4][NX], py[4][NX], pz[4][NX];
  ResSlab sy = {0.f, 0.f, 0.f}, sz = sy;
  bool in_y = false, in_z = false;
  unsigned in_x = 0u;               // bit q: plane i0 + q lies in an x slab
  float ghy = 0.f, ghz = 0.f, gey = 0.f, gez = 0.f;
  float xey = 0.f, xez = 0.f, xhy = 0.f, xhz = 0.f;     // x halo: E ahead, H behind
  unsigned snap_bits = 0u;
  const int m0 = in_tile ? row * rs + col : 0;   // this thread's cell in sh.e; + rs + 1 in sh.h

  // ---- LDS: fields, profiles, point operations, snapshots --------------------
  for (int t = tid; t < 3 * NX * kResPS; t += T) {
    (&sh.e[0][0][0])[t] = 0.f;
    (&sh.h[0][0][0])[t] = 0.f;
  }
  {
    const KParams& p = *pp;
#pragma unroll
    for (int q = 0; q < NX; ++q) {
      const int i = i0 + q, lx = i < p.cn[0] ? i : i - (p.nx - p.cn[1]);
      const bool xlo = i < p.cn[0], slab = i < p.nx && (xlo || lx >= 0);
      if (slab) in_x |= 1u << q;
      if (tid == q && i < p.nx) {
        sh.xprof[q] = slab ? make_float4(gld(xlo ? p.pb[0] : p.pb[1], lx),
                                         gld(xlo ? p.pc[0] : p.pc[1], lx),
                                         xlo ? p.cinv[0] : p.cinv[1], 0.f)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
        sh.gx[0][q] = GRADED ? gld(p.inv_h[0], i) : 0.f;
        sh.gx[1][q] = GRADED ? gld(p.inv_e[0], i) : 0.f;
      }
    }
  }
  if (tid < io.n_snap) sh.snap[tid] = io.snaps[tid];
  if (tid == 0) {
    sh.n_ops = 0;
    sh.bad = 0;
    sh.spin = io.spin;
  }
  __syncthreads();
  int op_lo = 0, op_n = 0;          // this thread's operations
  {
    // stable compaction of the block's operations (the plan checks the count)
    const KParams& p = *pp;
    for (int base = 0; base < p.n_ops; base += T) {
      const int t = base + tid;
      bool in = false;
      rfxh_point_op op;
      int own = 0;
      if (t < p.n_ops) {
        op = p.ops[t];
        const int i = (int)(op.cell / p.plane);
        const int r = (int)(op.cell - (long long)i * p.plane);
        const int oj = r / p.nz - by * ty, ok = r % p.nz - bz * tz;
        in = i >= i0 && i < i0 + NX && oj >= 0 && oj < ty && ok >= 0 && ok < tz;
        own = ok < sz_lo ? ty * n_in + oj * n_sl + ok
              : ok < sz_lo + n_in ? oj * n_in + ok - sz_lo
                                  : ty * n_in + oj * n_sl + ok - n_in;
        own = own * NX + i - i0;
      }
      const u64 bal = __ballot(in);
      const int w = tid >> 6, l = tid & 63;
      if (l == 0) sh.wcnt[w] = __popcll(bal);
      __syncthreads();
      int off = sh.n_ops + __popcll(bal & ((1ull << l) - 1ull));
      for (int u = 0; u < w; ++u) off += sh.wcnt[u];
      if (in && off < kResOps) {
        ResOp& d = sh.ops[off];
        d.own = own;
        d.kind = op.kind;
        d.comp = op.comp;
        d.slot = op.slot;
        d.d_par = op.d_par;
        d.loop[0] = op.loop[0];
        d.loop[1] = op.loop[1];
        d.loop[2] = op.loop[2];
      }
      __syncthreads();
      if (tid == 0) {
        int tot = sh.n_ops;
        for (int u = 0; u < (T + 63) / 64; ++u) tot += sh.wcnt[u];
        sh.n_ops = min(tot, kResOps);
      }
      __syncthreads();
    }
    // into the order of their threads (rank by counting: few, and once)
    const int n = sh.n_ops;
    ResOp mine;
    int rank = 0;
    if (tid < n) {
      mine = sh.ops[tid];
      for (int t = 0; t < n; ++t)
        rank += sh.ops[t].own < mine.own || (sh.ops[t].own == mine.own && t < tid);
    }
    __syncthreads();
    if (tid < n) sh.ops[rank] = mine;
    __syncthreads();
    for (int t = 0; t < n; ++t) {
      const int th = sh.ops[t].own / NX;
      op_lo += th < tid;
      op_n += th == tid;
    }
  }
  const int n_ops = __builtin_amdgcn_readfirstlane(sh.n_ops);
  const int stage = n_ops > 0 ? min(kResWave / n_ops, 64) : 64;

  // ---- halo words ------------------------------------------------------------
  const int per_q = ty + tz, n_yz = 2 * NX * per_q;
  constexpr unsigned kW = 8u * res_words(NX), kQ = 16u * kResEdge, kYZ = 16u * kResThreads;
  const unsigned half = (unsigned)n_wg * res_words(NX);     // one phase and parity
  const bool x_next = bx + 1 < io.ntx, y_next = by + 1 < io.nty, z_next = bz + 1 < io.ntz;
  const bool x_prev = bx > 0, y_prev = by > 0, z_prev = bz > 0;
  const int wx = io.ntz * io.nty, wy = io.ntz;          // workgroup strides along x, y
  // where a word goes in LDS (-1: this thread has no such word) and comes from
  // in a mailbox half (a thread without one reads its own mailbox, unused)
  int lds_e[kResWords], lds_h[kResWords];
  unsigned src_e[kResWords], src_h[kResWords];
#pragma unroll
  for (int m = 0; m < kResWords; ++m) {
    const KParams& p = *pp;
    const int w = tid + m * T;
    lds_e[m] = lds_h[m] = -1;
    src_e[m] = src_h[m] = (unsigned)wg * kW;
    if (w >= n_yz) continue;
    const int c = w & 1, r = w >> 1, q = r / per_q, pos = r - q * per_q;
    const unsigned at = kYZ + (unsigned)q * kQ + 16u * (unsigned)pos + 8u * (unsigned)c;
    const bool yw = pos < tz;
    const int comp = c == 0 ? 0 : yw ? 2 : 1;
    const int base = (comp * NX + q) * kResPS;
    if (yw ? y_next : z_next) {
      lds_e[m] = base + (yw ? ty * rs + pos : (pos - tz) * rs + tz);
      src_e[m] = (unsigned)(wg + (yw ? wy : 1)) * kW + at;
      // the first H update takes the neighbour's E from memory
      const int hi = i0 + q, hj = yw ? by * ty + ty : by * ty + pos - tz;
      const int hk = yw ? bz * tz + pos : bz * tz + tz;
      if (hi < p.nx && hj < p.ny && hk < p.nz) {
        const float* fp = comp == 0 ? io.f[0] : comp == 1 ? io.f[1] : io.f[2];
        (&sh.e[0][0][0])[lds_e[m]] =
            ldf(fp, ((unsigned)hi * (unsigned)p.ny + (unsigned)hj) * (unsigned)p.nz + (unsigned)hk);
      }
    }
    if (yw ? y_prev : z_prev) {
      lds_h[m] = base + (yw ? pos + 1 : (pos - tz + 1) * rs);
      src_h[m] = (unsigned)(wg - (yw ? wy : 1)) * kW + at;
    }
  }
  // The state and the memory to or from registers (out = false, true).
  auto state = [&](bool out, const int i0, const int j, const int k) {
    const KParams& p = *pp;
    const bool live = in_tile && j < p.ny && k < p.nz;
    const unsigned P = (unsigned)p.plane;
    const unsigned c0 = live ? (unsigned)i0 * P + (unsigned)j * (unsigned)p.nz + (unsigned)k : 0u;
    // a thread's cells all lie in the same y slab and the same z slab (or none)
    const int hj = j - (p.ny - p.cn[3]), hk = k - (p.nz - p.cn[5]);
    const bool ylo = j < p.cn[2], zlo = k < p.cn[4];
    const int ly = ylo ? j : hj, lz = zlo ? k : hk;
    const bool iy = live && (ylo || hj >= 0), iz = live && (zlo || hk >= 0);
    const unsigned ny_l = (unsigned)(ylo ? p.cn[2] : p.cn[3]);
    const unsigned nz_l = (unsigned)(zlo ? p.cn[4] : p.cn[5]);
    const unsigned y_at = (ylo ? io.foff[2] : io.foff[3]) +
                          ((unsigned)i0 * ny_l + (unsigned)ly) * (unsigned)p.nz + (unsigned)k;
    const unsigned z_at = (zlo ? io.foff[4] : io.foff[5]) +
                          ((unsigned)i0 * (unsigned)p.ny + (unsigned)j) * nz_l + (unsigned)lz;
    const unsigned y_st = ny_l * (unsigned)p.nz, z_st = (unsigned)p.ny * nz_l;
    const unsigned y_t = ylo ? io.fs[2] : io.fs[3], z_t = zlo ? io.fs[4] : io.fs[5];
    if (!out) {
      in_y = iy;
      in_z = iz;
      if (iy) {
        sy.b = gld(ylo ? p.pb[2] : p.pb[3], ly);
        sy.c = gld(ylo ? p.pc[2] : p.pc[3], ly);
        sy.inv = ylo ? p.cinv[2] : p.cinv[3];
      }
      if (iz) {
        sz.b = gld(zlo ? p.pb[4] : p.pb[5], lz);
        sz.c = gld(zlo ? p.pc[4] : p.pc[5], lz);
        sz.inv = zlo ? p.cinv[4] : p.cinv[5];
      }
      if (GRADED && live) {
        ghy = gld(p.inv_h[1], j);
        ghz = gld(p.inv_h[2], k);
        gey = gld(p.inv_e[1], j);
        gez = gld(p.inv_e[2], k);
      }
    }
#pragma unroll
    for (int q = 0; q < NX; ++q) {
      if (!out) {
        ex[q] = ey[q] = ez[q] = hx[q] = hy[q] = hz[q] = ca[q] = cb[q] = ce[q] = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t) px[t][q] = py[t][q] = pz[t][q] = 0.f;
      }
      const int i = i0 + q;
      if (!live || i >= p.nx) {
        if (!out) fl |= 7u << (4 * q);
        continue;
      }
      const unsigned c = c0 + (unsigned)q * P;
      // x slab of this plane: uniform over the workgroup
      const bool xlo = i < p.cn[0];
      const int lx = xlo ? i : i - (p.nx - p.cn[1]);
      const bool ix = xlo || lx >= 0;
      const unsigned x_at = (xlo ? io.foff[0] : io.foff[1]) +
                            ((unsigned)lx * (unsigned)p.ny + (unsigned)j) * (unsigned)p.nz +
                            (unsigned)k;
      const unsigned x_t = xlo ? io.fs[0] : io.fs[1];
      if (out) {
        stf(io.f[0], c, ex[q]);
        stf(io.f[1], c, ey[q]);
        stf(io.f[2], c, ez[q]);
        stf(io.f[3], c, hx[q]);
        stf(io.f[4], c, hy[q]);
        stf(io.f[5], c, hz[q]);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (ix) stf(io.psi, x_at + t * x_t, px[t][q]);
          if (iy) stf(io.psi, y_at + q * y_st + t * y_t, py[t][q]);
          if (iz) stf(io.psi, z_at + q * z_st + t * z_t, pz[t][q]);
        }
        continue;
      }
      ex[q] = ldf(io.f[0], c);
      ey[q] = ldf(io.f[1], c);
      ez[q] = ldf(io.f[2], c);
      hx[q] = ldf(io.f[3], c);
      hy[q] = ldf(io.f[4], c);
      hz[q] = ldf(io.f[5], c);
      const float4 co = gld(p.ecoef, (int)ldu16(p.mat, c));
      ca[q] = co.x;
      cb[q] = co.y;
      ce[q] = co.z;
      unsigned f = __float_as_uint(co.w) & 7u;
      if ((p.pec_axes & 1) && (i == 0 || i == p.nx - 1)) f |= RFXH_ZERO_EY | RFXH_ZERO_EZ;
      if ((p.pec_axes & 2) && (j == 0 || j == p.ny - 1)) f |= RFXH_ZERO_EX | RFXH_ZERO_EZ;
      if (p.pec_axes & 4) {
        if (k == 0 || k == p.nz - 1) f |= RFXH_ZERO_EX | RFXH_ZERO_EY;
        if (k == p.nz - 1) f |= RFXH_ZERO_EZ;
      }
      fl |= f << (4 * q);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (ix) px[t][q] = ldf(io.psi, x_at + t * x_t);
        if (iy) py[t][q] = ldf(io.psi, y_at + q * y_st + t * y_t);
        if (iz) pz[t][q] = ldf(io.psi, z_at + q * z_st + t * z_t);
      }
    }
    if (!out && live && bx + 1 < io.ntx) {
      xey = ldf(io.f[1], c0 + (unsigned)NX * P);
      xez = ldf(io.f[2], c0 + (unsigned)NX * P);
    }
  };
  // (after the set-up above, whose temporaries would not fit beside it)
  state(false, i0, j, k);
#pragma unroll
  for (int q = 0; q < NX; ++q)
    if (in_tile) {
      sh.e[0][q][m0] = ex[q];
      sh.e[1][q][m0] = ey[q];
      sh.e[2][q][m0] = ez[q];
    }
  // snapshots this thread's cells can belong to
  for (int t = 0; t < io.n_snap; ++t) {
    const ResSnap& s = sh.snap[t];
    const int a = s.axis == 0 ? j : i0, b = s.axis == 2 ? j : k;
    bool hit = in_tile && b >= s.lo2 && b < s.hi2;
    if (s.axis == 0) hit = hit && a >= s.lo1 && a < s.hi1 && s.index >= i0 && s.index < i0 + NX;
    else hit = hit && a + NX > s.lo1 && a < s.hi1 && (s.axis == 1 ? j : k) == s.index;
    if (hit) snap_bits |= 1u << t;
  }
  // Fetch the halo of one phase: the tagged words of `src` into LDS and the
  // two x words at xsrc into a, b.  Every lane loads every word, so that the
  // loads are in flight together with no branch between them.
  auto fetch = [&](const u64* from, unsigned tag, const int (&dst)[kResWords],
                   const unsigned (&src)[kResWords], float* lds, unsigned need_x, unsigned xsrc,
                   float& a, float& b) {
    u64 v[kResWords], va, vb;
    for (int n = 0;;) {
      // (opaque: 32-bit offsets from the scalar base, not 64-bit addresses)
      unsigned ox = xsrc;
      __asm__ volatile("" : "+v"(ox));
      va = res_ld(from, ox);
      vb = res_ld(from, ox + 8u);
#pragma unroll
      for (int m = 0; m < kResWords; ++m) {
        unsigned o = src[m];
        __asm__ volatile("" : "+v"(o));
        v[m] = res_ld(from, o);
      }
      unsigned off = (((unsigned)(va >> 32) ^ tag) | ((unsigned)(vb >> 32) ^ tag)) & need_x;
#pragma unroll
      for (int m = 0; m < kResWords; ++m)
        off |= ((unsigned)(v[m] >> 32) ^ tag) & (unsigned)~(dst[m] >> 31);
      if (off == 0u) break;
      // (the limit from LDS and only at a look: a kernel argument in this loop
      // cost 2 % of a 28^3 step, a store to `stop` 1.6 %)
      if (++n % kResLook == 0 &&
          (sh.bad || n >= sh.spin ||
           __hip_atomic_load(io.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
        sh.bad = 1;
        break;
      }
    }
    a = need_x ? __uint_as_float((unsigned)va) : 0.f;
    b = need_x ? __uint_as_float((unsigned)vb) : 0.f;
#pragma unroll
    for (int m = 0; m < kResWords; ++m)
      if (dst[m] >= 0) lds[dst[m]] = __uint_as_float((unsigned)v[m]);
  };
  // the workgroup's barrier for LDS alone: the mailbox stores stay in flight
  // (__syncthreads would wait for their acknowledgement)
  auto lds_barrier = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  // Loop-invariant scalars.  What differs between lanes is kept as bits of one
  // register and tested where it is used: as lane masks in scalar registers
  // these conditions spilled, with the parameters they pushed out.
  const float ch = pp->ch_all, inv_h0 = pp->inv_h0, inv_e0 = pp->inv_e0;
  const unsigned roles = (in_tile ? 1u : 0u) | (in_tile && x_next ? 2u : 0u) |
                         (in_tile && x_prev ? 4u : 0u) |
                         (in_tile && row == ty - 1 && y_next ? 8u : 0u) |
                         (in_tile && col == tz - 1 && z_next ? 16u : 0u) |
                         (in_tile && row == 0 && y_prev ? 32u : 0u) |
                         (in_tile && col == 0 && z_prev ? 64u : 0u) | (in_y ? 128u : 0u) |
                         (in_z ? 256u : 0u);
  const unsigned need_h = (roles & 4u) ? ~0u : 0u, need_e = (roles & 2u) ? ~0u : 0u;
  const unsigned xs_h = (unsigned)(need_h ? wg - wx : wg) * kW + 16u * (unsigned)tid;
  const unsigned xs_e = (unsigned)(need_e ? wg + wx : wg) * kW + 16u * (unsigned)tid;
  const int n_steps = io.n_steps;
  __syncthreads();

  bool bad = false;
  unsigned tag = io.tag0;
  int w_base = 0, w_next = 0;           // first step of the staged source values, of the next ones
  for (int n = 0; n < n_steps; ++n) {
    const int par = n & 1;
    u64* const box_h = io.box + (unsigned)par * half;
    u64* const box_e = io.box + (unsigned)(2 + par) * half;
    // own words; opaque to the compiler, which would otherwise keep the
    // address of each of a thread's stores in a register through the loop
    unsigned out_x = (unsigned)wg * kW + 16u * (unsigned)tid;
    unsigned out_y = (unsigned)wg * kW + kYZ + 16u * (unsigned)col;
    unsigned out_z = (unsigned)wg * kW + kYZ + 16u * (unsigned)(tz + row);
    unsigned role = roles;
    __asm__ volatile("" : "+v"(out_x), "+v"(out_y), "+v"(out_z), "+v"(role));
    const unsigned tag_h = ++tag, tag_e = ++tag;
    if (n_ops > 0 && n == w_next) {
      // the source values of the next `stage` steps
      w_base = n;
      w_next = n + stage;
      for (int t = tid; t < n_ops * stage; t += T) {
        const int s = t / n_ops, o = t - s * n_ops;
        if (sh.ops[o].kind == RFXH_OP_INJECT && n + s < n_steps)
          sh.w[t] = io.src_wave[(io.step0 + n + s) * io.n_src + sh.ops[o].slot];
      }
    }
    // ---- H (cells outside the grid stay zero: so do their forward neighbours)
#pragma unroll
    for (int q0 = 0; q0 < NX; q0 += G) {
      float dzy[G], dyz[G], dxz[G], dzx[G], dyx[G], dxy[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int q = q0 + u;
        dxy[u] = sh.e[0][q][m0 + rs];
        dzy[u] = sh.e[2][q][m0 + rs];
        dxz[u] = sh.e[0][q][m0 + 1];
        dyz[u] = sh.e[1][q][m0 + 1];
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int q = q0 + u;
        dxy[u] -= ex[q];
        dzy[u] -= ez[q];
        dxz[u] -= ex[q];
        dyz[u] -= ey[q];
        dzx[u] = (q + 1 < NX ? ez[q + 1 < NX ? q + 1 : q] : xez) - ez[q];
        dyx[u] = (q + 1 < NX ? ey[q + 1 < NX ? q + 1 : q] : xey) - ey[q];
        const float ix = GRADED ? sh.gx[0][q] : inv_h0;
        const float iy = GRADED ? ghy : inv_h0, iz = GRADED ? ghz : inv_h0;
        hx[q] = __builtin_fmaf(-ch, res_curl(iy, dzy[u], iz, dyz[u]), hx[q]);
        hy[q] = __builtin_fmaf(-ch, res_curl(iz, dxz[u], ix, dzx[u]), hy[q]);
        hz[q] = __builtin_fmaf(-ch, res_curl(ix, dyx[u], iy, dxy[u]), hz[q]);
      }
      if (in_x) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int q = q0 + u;
          if (!((in_x >> q) & 1u)) continue;
          const float4 pr = sh.xprof[q];
          const ResSlab s = {pr.x, pr.y, pr.z};
          float d0, d1;
          res_slab(s, ch, dzx[u], dyx[u], px[0][q], px[1][q], d0, d1);
          hy[q] += d0;
          hz[q] -= d1;
        }
      }
      if (role & 128u) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int q = q0 + u;
          float d0, d1;
          res_slab(sy, ch, dzy[u], dxy[u], py[0][q], py[1][q], d0, d1);
          hx[q] -= d0;
          hz[q] += d1;
        }
      }
      if (role & 256u) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int q = q0 + u;
          float d0, d1;
          res_slab(sz, ch, dyz[u], dxz[u], pz[0][q], pz[1][q], d0, d1);
          hx[q] += d0;
          hy[q] -= d1;
        }
      }
    }
    // ---- H of the high faces to the workgroups ahead, own H to LDS
    if (role & 2u) res_st2(box_h, out_x, hy[NX - 1], hz[NX - 1], tag_h);
    if (role & 8u) {
#pragma unroll
      for (int q = 0; q < NX; ++q) {
        res_st2(box_h, out_y + (unsigned)q * kQ, hx[q], hz[q], tag_h);
      }
    }
    if (role & 16u) {
#pragma unroll
      for (int q = 0; q < NX; ++q) {
        res_st2(box_h, out_z + (unsigned)q * kQ, hx[q], hy[q], tag_h);
      }
    }
    if (role & 1u) {
#pragma unroll
      for (int q = 0; q < NX; ++q) {
        sh.h[0][q][m0 + rs + 1] = hx[q];
        sh.h[1][q][m0 + rs + 1] = hy[q];
        sh.h[2][q][m0 + rs + 1] = hz[q];
      }
    }
    fetch(box_h, tag_h, lds_h, src_h, &sh.h[0][0][0], need_h, xs_h, xhy, xhz);
    lds_barrier();
    // ---- E
#pragma unroll
    for (int q0 = 0; q0 < NX; q0 += G) {
      float dzy[G], dyz[G], dxz[G], dzx[G], dyx[G], dxy[G];
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int q = q0 + u;
        dxy[u] = sh.h[0][q][m0 + 1];
        dzy[u] = sh.h[2][q][m0 + 1];
        dxz[u] = sh.h[0][q][m0 + rs];
        dyz[u] = sh.h[1][q][m0 + rs];
      }
#pragma unroll
      for (int u = 0; u < G; ++u) {
        const int q = q0 + u;
        dxy[u] = hx[q] - dxy[u];
        dzy[u] = hz[q] - dzy[u];
        dxz[u] = hx[q] - dxz[u];
        dyz[u] = hy[q] - dyz[u];
        dzx[u] = hz[q] - (q > 0 ? hz[q > 0 ? q - 1 : 0] : xhz);
        dyx[u] = hy[q] - (q > 0 ? hy[q > 0 ? q - 1 : 0] : xhy);
        const float ix = GRADED ? sh.gx[1][q] : inv_e0;
        const float iy = GRADED ? gey : inv_e0, iz = GRADED ? gez : inv_e0;
        {
#pragma clang fp contract(off)
          ex[q] = __builtin_fmaf(ex[q], ca[q], res_curl(iy, dzy[u], iz, dyz[u]) * cb[q]);
          ey[q] = __builtin_fmaf(ey[q], ca[q], res_curl(iz, dxz[u], ix, dzx[u]) * cb[q]);
          ez[q] = __builtin_fmaf(ez[q], ca[q], res_curl(ix, dyx[u], iy, dxy[u]) * cb[q]);
        }
      }
      if (in_x) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int q = q0 + u;
          if (!((in_x >> q) & 1u)) continue;
          const float4 pr = sh.xprof[q];
          const ResSlab s = {pr.x, pr.y, pr.z};
          float d0, d1;
          res_slab(s, ce[q], dzx[u], dyx[u], px[2][q], px[3][q], d0, d1);
          ey[q] -= d0;
          ez[q] += d1;
        }
      }
      if (role & 128u) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int q = q0 + u;
          float d0, d1;
          res_slab(sy, ce[q], dzy[u], dxy[u], py[2][q], py[3][q], d0, d1);
          ex[q] += d0;
          ez[q] -= d1;
        }
      }
      if (role & 256u) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const int q = q0 + u;
          float d0, d1;
          res_slab(sz, ce[q], dyz[u], dxz[u], pz[2][q], pz[3][q], d0, d1);
          ex[q] -= d0;
          ey[q] += d1;
        }
      }
    }
    if (fl) {
#pragma unroll
      for (int q = 0; q < NX; ++q) {
        const unsigned f = fl >> (4 * q);
        ex[q] = (f & RFXH_ZERO_EX) ? 0.f : ex[q];
        ey[q] = (f & RFXH_ZERO_EY) ? 0.f : ey[q];
        ez[q] = (f & RFXH_ZERO_EZ) ? 0.f : ez[q];
      }
    }
    for (int o = op_lo; o < op_lo + op_n; ++o) {
      // (point_ops; H of the cell and behind it from LDS, E from registers)
      const ResOp op = sh.ops[o];
      const int c = op.comp, oq = op.own - tid * NX, at = m0 + rs + 1;
      if (op.kind == RFXH_OP_INJECT) {
        const float w = sh.w[(n - w_base) * n_ops + o];
#pragma unroll
        for (int q = 0; q < NX; ++q) {
          if (q != oq) continue;
          if (c == 0) ex[q] += w;
          else if (c == 1) ey[q] += w;
          else ez[q] += w;
        }
        continue;
      }
      float e0 = ex[0], e1 = ey[0], e2 = ez[0];
#pragma unroll
      for (int q = 1; q < NX; ++q)
        if (q == oq) {
          e0 = ex[q];
          e1 = ey[q];
          e2 = ez[q];
        }
      const float h0 = sh.h[0][oq][at], h1 = sh.h[1][oq][at], h2 = sh.h[2][oq][at];
      if (op.kind == RFXH_OP_PORT) {
        const float v = -pick3(c, e0, e1, e2) * op.d_par;
        const float hx_j = sh.h[0][oq][at - rs], hz_j = sh.h[2][oq][at - rs];
        const float hx_k = sh.h[0][oq][at - 1], hy_k = sh.h[1][oq][at - 1];
        const float hy_i = oq > 0 ? sh.h[1][max(oq - 1, 0)][at] : xhy;
        const float hz_i = oq > 0 ? sh.h[2][max(oq - 1, 0)][at] : xhz;
        float cur;
        if (c == 2)
          cur = (h1 - hy_i) * op.loop[1] - (h0 - hx_j) * op.loop[0];
        else if (c == 0)
          cur = (h2 - hz_j) * op.loop[2] - (h1 - hy_k) * op.loop[1];
        else
          cur = (h0 - hx_k) * op.loop[0] - (h2 - hz_i) * op.loop[2];
        float* const out = io.port_out + ((io.step0 + n) * io.n_port + op.slot) * 2;
        out[0] = v;
        out[1] = cur;
      } else {
        io.probe_out[(io.step0 + n) * io.n_probe + op.slot] =
            c < 3 ? pick3(c, e0, e1, e2) : pick3(c - 3, h0, h1, h2);
      }
    }
    const bool last = n + 1 == n_steps;
    if (!last) {
      // ---- E of the low faces to the workgroups behind, own E to LDS
      if (role & 4u) res_st2(box_e, out_x, ey[0], ez[0], tag_e);
      if (role & 32u) {
#pragma unroll
        for (int q = 0; q < NX; ++q) {
          res_st2(box_e, out_y + (unsigned)q * kQ, ex[q], ez[q], tag_e);
        }
      }
      if (role & 64u) {
#pragma unroll
        for (int q = 0; q < NX; ++q) {
          res_st2(box_e, out_z + (unsigned)q * kQ, ex[q], ey[q], tag_e);
        }
      }
      if (role & 1u) {
#pragma unroll
        for (int q = 0; q < NX; ++q) {
          sh.e[0][q][m0] = ex[q];
          sh.e[1][q][m0] = ey[q];
          sh.e[2][q][m0] = ez[q];
        }
      }
    }
    if (snap_bits) {
      // after the faces are on their way: nobody waits for these
      for (int t = 0; t < io.n_snap; ++t) {
        if (!((snap_bits >> t) & 1u)) continue;
        const ResSnap& s = sh.snap[t];
        const int v = (s.axis == 2 ? j : k) - s.lo2;
        float* const o = s.out + (long long)n * s.ncomp * s.npts + v;
#pragma unroll
        for (int q = 0; q < NX; ++q) {
          const int i = i0 + q;
          if (s.axis == 0 ? i != s.index : (i < s.lo1 || i >= s.hi1)) continue;
          float* const oq = o + (long long)((s.axis == 0 ? j : i) - s.lo1) * s.n2;
          // H of the plane behind (the plane itself at index 0)
          const int at = m0 + rs + 1, back = s.axis == 1 ? at - rs : at - 1;
          const bool self = s.index == 0;
          for (int c = 0; c < s.ncomp; ++c) {
            const int cc = s.comp[c];
            float x = cc < 3 ? pick3(cc, ex[q], ey[q], ez[q]) : pick3(cc - 3, hx[q], hy[q], hz[q]);
            if (s.avg && cc >= 3) {
              const float b = self ? x
                              : s.axis == 0 ? (cc == 4 ? (q > 0 ? hy[q > 0 ? q - 1 : 0] : xhy)
                                                       : (q > 0 ? hz[q > 0 ? q - 1 : 0] : xhz))
                                            : sh.h[cc - 3][q][back];
              x = (b + x) * 0.5f;
            }
            oq[c * s.npts] = x;
          }
        }
      }
    }
    if (last) break;
    fetch(box_e, tag_e, lds_e, src_e, &sh.e[0][0][0], need_e, xs_e, xey, xez);
    lds_barrier();
    if ((n & 31) == 31) {
      // (the second barrier: no wavefront is at its next wait, which may set
      // `bad`, before all have read it, so all leave at the same step)
      bad = sh.bad;
      lds_barrier();
      if (bad) break;
    }
  }
  bad = bad || sh.bad;
  if (bad && tid == 0)
    __hip_atomic_store(io.stop, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // (opaque positions: the addresses of the way in would stay in registers)
  int oi = i0, oj = j, ok = k;
  __asm__ volatile("" : "+v"(oj), "+v"(ok), "+s"(oi) : : "memory");
  state(true, oi, oj, ok);
}

// Adds the staged steps [0, cnt) of a launch that started at step n0 to the
// float64 accumulators of one plane, step by step in order as dft_fold and
// flux_fold do; one thread per (point, component, group of kFoldF
// frequencies).  twe: twiddles of components 0 and 1, twh: of 2 and 3.
__global__ __launch_bounds__(256) void k_res_fold(const float* ring, int ncomp, long long npts,
                                                  const double2* twe, const double2* twh,
                                                  double2* acc, int nf, long long n0, int cnt) {
  const long long pidx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (pidx >= npts) return;
  const int t = (int)blockIdx.y, f0 = (int)blockIdx.z * kFoldF;
  const double2* tw = t < 2 ? twe : twh;
  double2* a = acc + (long long)t * nf * npts + pidx;
  double2 cur[kFoldF];
#pragma unroll
  for (int u = 0; u < kFoldF; ++u)
    cur[u] = f0 + u < nf ? a[(long long)(f0 + u) * npts] : make_double2(0.0, 0.0);
  for (int m = 0; m < cnt; ++m) {
    const double x = (double)ring[((long long)m * ncomp + t) * npts + pidx];
#pragma unroll
    for (int u = 0; u < kFoldF; ++u) {
      if (f0 + u >= nf) break;
      const double2 w = tw[(n0 + m) * nf + f0 + u];
      cur[u].x += w.x * x;
      cur[u].y += w.y * x;
    }
  }
#pragma unroll
  for (int u = 0; u < kFoldF; ++u)
    if (f0 + u < nf) a[(long long)(f0 + u) * npts] = cur[u];
}

// After a run whose launches gave up somewhere: its fields, probe and port rows
// and the accumulators become NaN, and the host's word is set.
struct ResOut {
  const unsigned* stop;
  unsigned* status;                 // pinned host memory
  float* f[6];
  long long cells;
  float *probe, *port;              // first row of the run
  long long n_probe, n_port;        // floats of its rows
  const MonEntry* mon;
  int n_mon;
};

__global__ __launch_bounds__(256) void k_res_check(ResOut o) {
  if (__hip_atomic_load(o.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) return;
  const long long t0 = (long long)blockIdx.x * 256 + threadIdx.x, T = (long long)gridDim.x * 256;
  const float nan = __uint_as_float(0x7fc00000u);
  for (long long t = t0; t < o.cells; t += T)
    for (int c = 0; c < 6; ++c) o.f[c][t] = nan;
  for (long long t = t0; t < o.n_probe; t += T) o.probe[t] = nan;
  for (long long t = t0; t < o.n_port; t += T) o.port[t] = nan;
  for (int e = 0; e < o.n_mon; ++e) {
    const MonEntry& m = o.mon[e];
    const long long n = m.flux ? 4LL * m.f.nf * m.f.n1 * m.f.n2 : (long long)m.p.nf * m.p.n1 * m.p.n2;
    double2* const acc = m.flux ? m.f.acc : m.p.acc;
    for (long long t = t0; t < n; t += T) acc[t] = make_double2((double)nan, (double)nan);
  }
  if (t0 == 0) __hip_atomic_store(o.status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
