// Persistent kernels of the MI355X tdse engine (gfx950): whole attempts in
// one cooperative launch.
//
//   k_rows_begin     unsets the exchange buffers, saves the state.
//   k_rows_run       small systems, also a few pulses: workgroups own rows.
//   k_tiles_run      larger systems: workgroups own tiles and rows.
//
// Compiled without the machine-code loop-invariant motion, which would hold
// the constants of the controller's and the field's functions in registers
// through the whole run (k_tiles_run: 46 spilled registers with it).
#include "device.hpp"

namespace mpci {

// ---------------------------------------------------------------------
// Persistent row kernel: whole attempts of one pulse in one cooperative
// launch (every workgroup resident, one per compute unit).  A workgroup owns
// up to 64 rows of one block.  Four waves compute, a quad each (two or four
// when a workgroup has more rows): the first kRwReg chunks of a quad's part
// of the row store stay in registers for the whole launch, further ones in
// LDS, the rest comes from L2; the rows' 13 stage derivatives stay in LDS.
// The other four waves poll the neighbour blocks' stage input into one of
// two LDS copies, so a stage has one workgroup barrier and one exchange.
//
// What bounds it: latency.  Per stage (4 x 198, clock64): about 0.9 us from
// a store to its reader, 0.4 us for the coupling sums and their lane
// reduction, 0.3 us for the stage algebra; a launch per stage took 5.7 us.
// Whole attempts 83 -> 31.6 us (4 x 198), 105 -> 34.9 us (6 x 300), 165 ->
// 72 us (blocks 1201, 1333, 997, where the neighbours' 2198 rows of 16
// bytes per workgroup weigh as much as the dipoles).  Tried: coupling sums
// split over all eight waves with a second barrier and an LDS sum (42 and
// 49 us; a wave64 instruction takes four cycles, and eight waves reducing 32
// sums each issue more of them than four waves reducing eight), every wave
// polling and storing (47 us: a poll waits for the acknowledgement of the
// stores before it), 16 waves (register spills).
//
// A batch (kMany): the device holds ngrp groups of workgroups, each with all
// rows, and a group runs some of the pulses, up to kRwSlots at a time: a
// stage of each in turn, so that a pulse's exchange runs behind the others'
// sums.  Pulses stay independent: each has its exchange buffers, its step
// control (a polling wave each) and its attempts.  Per attempt of all pulses,
// against the batched launches (13 GEMM and 13 stage launches of 5 to 14 us
// each whatever they hold): 300 x 6, P = 5 164 -> 62 us; 198 x 4, P = 16 145
// -> 78 us; 60 x 8, P = 5 128 -> 28 us.  One launch may hold several batches
// (RowRuns), each with workgroups of its own.  A further pulse of a group costs
// about 20 us, 1.5 us a stage: the computing waves' tableau sums, coupling
// sums and stage algebra.  Fewer, larger groups (32 to 64 rows a workgroup)
// were slower from P = 2 on (300 x 6, P = 5: 98 to 141 us).
//
// Exchange.  xb holds four copies of the state; stage g (counted over the
// launch) uses copy g % 4.  An unset component holds kUnset, a signalling
// NaN that no arithmetic produces (a raw copy of it is quieted).  The owner
// of a row stores its stage input with device-scope (write-through) stores;
// a reader polls the rows it needs with device-scope loads, 16 bytes at a
// time, until both components are set, so the data is its own flag.  A
// workgroup that has read every neighbour row of stage g knows that all its
// readers have finished with copy (g + 3) % 4 (they published stage g after
// reading stage g - 1), and unsets its own rows there; those stores have
// landed before it publishes stage g + 2, ahead of any poll of that copy for
// stage g + 3.  The step control needs every row's error and norm: quads
// exchange them the same way (rb, three copies by attempt), one wave of every
// workgroup reduces them in k_finalize's order and runs the controller, with
// the same bits everywhere.
//
// Every wait is bounded: past limit_ms a workgroup sets abort_flag and
// leaves, the others see the flag; the host then restores the state saved
// by k_rows_begin and runs the attempts with one launch per stage.
// ---------------------------------------------------------------------
constexpr unsigned long long kUnset = 0x7FF4C0DEFACE0FF5ull;
template <int V>
struct Int {
  static constexpr int value = V;
};
constexpr int kXbCopies = 4;   // copies of the state in exchange
constexpr int kScDevice = 16;  // sc1: device-scope load / store

typedef unsigned uv4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bool is_unset(double v) {
  return (unsigned long long)__double_as_longlong(v) == kUnset;
}

__device__ __forceinline__ double2 dev_load(__amdgpu_buffer_rsrc_t r,
                                            unsigned byte) {
  const uv4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)byte, 0,
                                                      kScDevice);
  return make_double2(__hiloint2double((int)v.y, (int)v.x),
                      __hiloint2double((int)v.w, (int)v.z));
}

__device__ __forceinline__ void dev_store(__amdgpu_buffer_rsrc_t r,
                                          unsigned byte, double2 x) {
  const uv4 v = {(unsigned)__double2loint(x.x), (unsigned)__double2hiint(x.x),
                 (unsigned)__double2loint(x.y), (unsigned)__double2hiint(x.y)};
  __builtin_amdgcn_raw_buffer_store_b128(v, r, (int)byte, 0, kScDevice);
}

__device__ __forceinline__ void dev_store1(__amdgpu_buffer_rsrc_t r,
                                           unsigned byte, double x) {
  typedef unsigned uv2 __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(
      uv2{(unsigned)__double2loint(x), (unsigned)__double2hiint(x)}, r,
      (int)byte, 0, kScDevice);
}

// a value as published: never kUnset
__device__ __forceinline__ double publishable1(double v) {
  return is_unset(v) ? __longlong_as_double((long long)(kUnset | (1ull << 51)))
                     : v;
}
__device__ __forceinline__ double2 publishable(double2 v) {
  return make_double2(publishable1(v.x), publishable1(v.y));
}

// Unsets the exchange buffers and saves the states and control records.
__global__ __launch_bounds__(256) void k_rows_begin(
    double2 *xb, int nxb, double2 *pb, int npb, double2 *rb, int nrb,
    const double2 *X, int NP, double2 *Xsave, Ctl *ctl, int P,
    int *abort_flag, int *arrived) {
  const double u = __longlong_as_double((long long)kUnset);
  const double2 unset = make_double2(u, u);
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < nxb) xb[i] = unset;
  if (i < npb) pb[i] = unset;
  if (i < nrb) rb[i] = unset;
  if (i < NP) Xsave[i] = X[i];
  if (i < P) ctl[P + i] = ctl[i];
  if (i == 0) {
    *abort_flag = 0;
    *arrived = 0;
  }
}

// A launch that is not cooperative begins only when all its workgroups run:
// each (one thread of it) reports and waits, start_ms at most.  False: this
// one waited in vain, and all of them leave.
__device__ __forceinline__ bool all_started(int *arrived, int *abort_flag,
                                            int start_ms) {
  __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  const long long t0 = wall_clock64();
  while (__hip_atomic_load(arrived, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT) < (int)gridDim.x) {
    if (__hip_atomic_load(abort_flag, __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT) != 0)
      return false;
    if (wall_clock64() - t0 > (long long)start_ms * 100000) {
      __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
    __builtin_amdgcn_s_sleep(8);
  }
  return true;
}

// Workgroup blk of run a.
template <int kQ, bool kMany>
__device__ __forceinline__ void rows_run(const RowRun &a, int blk) {
  const SysDesc *__restrict__ dp = a.d;
  const RowDesc *__restrict__ rp = a.rows;
  const double *__restrict__ Dq = a.Dq;
  // chunks of a quad kept in registers: one quad a wave leaves room for them
  constexpr int kReg = kQ == 1 ? kRwReg : 0;
  static_assert(!kMany || kQ == 1, "several slots: a quad a wave");
  constexpr int kSlots = kMany ? kRwSlots : 1;
  const SysDesc &d = *dp;
  // group grp of nwg workgroups runs pulses grp, grp + ngrp, .., nslot of
  // them at a time, a stage of each in turn
  const int grp = blk / a.nwg, wgi = blk - grp * a.nwg;
  const RowWg g = a.wg[wgi];
  const int attempts =
      g.quit > 0 && grp == a.ngrp - 1 ? g.quit - 1 : a.attempts;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int L = g.L, gauge = d.gauge;
  const int n0 = L > 0 ? d.off[L] - d.off[L - 1] : 0;
  const int n1 = L + 1 < d.nb ? d.off[L + 2] - d.off[L + 1] : 0;
  const int nch0 = (n0 + 63) >> 6, nch = nch0 + ((n1 + 63) >> 6);
  const int nchp = (nch + 3) & ~3;  // whole groups of four chunks
  const int nx = n0 + n1;
  const int nq = (g.nrows + kRwQuad - 1) / kRwQuad, nr4 = nq * kRwQuad;

  // LDS: two copies of the neighbours' stage input (zero padded to whole
  // groups of chunks); per slot the 13 stage derivatives, the state and the
  // stage input of the own rows; the resident chunks of the row store
  // ([quad][chunk])
  extern __shared__ __align__(16) unsigned char smem[];
  double2 *xs0 = reinterpret_cast<double2 *>(smem);
  double2 *own_rows = xs0 + 2 * nchp * 64;
  const int slot_n = (kStages + 2) * nr4;
  const unsigned nslot = kMany ? (unsigned)a.nslot : 1u;
  double2 *Dl = own_rows + nslot * slot_n;
  __shared__ Ctl cl[kSlots];
  __shared__ double2 en[kSlots][kRwMaxRows / kRwQuad];
  __shared__ int stop;
  // row s < 12: a_{s+1,j}; rows 12, 13: b, b - bhat
  __shared__ double coef[kStages + 1][kStages];

  const unsigned N = (unsigned)a.N, NQ = (unsigned)a.nquad;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.xb + (long long)grp * nslot * kXbCopies * N), (short)0,
      (int)(nslot * kXbCopies * N * 16u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.rb + (long long)grp * nslot * 3 * NQ), (short)0,
      (int)(nslot * 3u * NQ * 16u), 0x00020000);
  constexpr unsigned kOut = 0x80000000u;  // beyond any buffer range
  const double u_ = __longlong_as_double((long long)kUnset);
  const double2 unset = make_double2(u_, u_);

  if (t == 0) {
    stop = 0;
    if (a.limit_ms < 0) {  // no wait at all
      stop = 1;
      __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    } else if (a.start_ms > 0 &&
               !all_started(a.arrived, a.abort_flag, a.start_ms)) {
      stop = 1;
    }
  }
  if (t < (kStages + 1) * kStages) {
    const int s = t / kStages, j = t - s * kStages;
    coef[s][j] = s < kStages - 1 ? cA[s + 1][j] : s == kStages - 1 ? cB[j] : cDB[j];
  }
  for (int i = t; i < 2 * nchp * 64; i += kRwThreads)
    xs0[i] = make_double2(0.0, 0.0);
  const double2 *D2 = reinterpret_cast<const double2 *>(Dq + rp->q_off[L]) +
                      (long long)(g.row0 / kRwQuad) * nch * 128;
  for (int i = t; i < nq * g.nlds * 128; i += kRwThreads) {
    const int qc = i >> 7, q = qc / g.nlds, c = qc - q * g.nlds;
    const int ch = kReg + c;
    if (ch < nch) Dl[i] = D2[((long long)q * nch + ch) * 128 + (i & 127)];
  }
  __syncthreads();
  if (stop) return;  // uniform

  // true once the wait has to be given up (looked at now and then)
  long long t_wait = 0;
  auto give_up = [&](int tries) -> bool {
    if ((tries & 63) != 0) return false;
    const long long now = wall_clock64();
    if (tries == 64) t_wait = now;
    const bool late = now - t_wait > (long long)a.limit_ms * 100000;
    if (late)
      __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return late || __hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT) != 0;
  };

  // exchange copies, two bits a slot: of the coming attempt's stage 0 (13
  // stages on, the next attempt's is the next one) and of its reduction
  static_assert(kXbCopies == 4 && kStages % 4 == 1, "");
  unsigned xcopy = 0, rcopy = 0;
  auto bits2 = [](unsigned v, int b) { return (v >> (2 * b)) & 3u; };
  // the slots whose pulse is not finished, and their copies moved on
  auto live_slots = [&](int ns) {
    if (!kMany) return cl[0].done ? 0u : 1u;
    unsigned m = 0;
    for (int b = 0; b < ns; ++b)
      if (!cl[b].done) m |= 1u << b;
    return (unsigned)__builtin_amdgcn_readfirstlane((int)m);
  };
  auto advance = [&](unsigned act) {
    for (unsigned m = act; m; m &= m - 1) {
      const int b = kMany ? __builtin_ctz(m) : 0;
      const unsigned x1 = (bits2(xcopy, b) + 1) & 3u;
      const unsigned r1 = bits2(rcopy, b) == 2 ? 0u : bits2(rcopy, b) + 1;
      xcopy = (xcopy & ~(3u << (2 * b))) | (x1 << (2 * b));
      rcopy = (rcopy & ~(3u << (2 * b))) | (r1 << (2 * b));
    }
  };
  int par = 0;  // LDS copy of the coming stage's input
  if (w >= kRwCompute) {
    // ================= the polling waves =================
    const int tp = t - 64 * kRwCompute;
    constexpr int kPoll = kRwThreads - 64 * kRwCompute;
    const int row_lo = L > 0 ? d.off[L - 1] : 0;
    const int row_up = L + 1 < d.nb ? d.off[L + 1] : 0;
    const bool negate = gauge == 0;
    // U rows per thread, from slot u0 on, of exchange copy b into xs, all
    // in flight, polled until set
    auto poll = [&](unsigned b, double2 *xs, int u0, auto width) {
      constexpr int U = decltype(width)::value;
      unsigned miss = 0, off[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = (u0 + u) * kPoll + tp;
        if (i < nx) miss |= 1u << u;
        off[u] =
            (b * N + (unsigned)(i < n0 ? row_lo + i : row_up + i - n0)) * 16u;
      }
      for (int tries = 1; miss; ++tries) {
        double2 r[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
          r[u] = dev_load(rx, (miss >> u) & 1u ? off[u] : kOut);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (((miss >> u) & 1u) && !is_unset(r[u].x) && !is_unset(r[u].y)) {
            const int i = (u0 + u) * kPoll + tp;
            const bool up = i >= n0;
            xs[up ? nch0 * 64 + i - n0 : i] =
                up && negate ? make_double2(-r[u].x, -r[u].y) : r[u];
            miss &= ~(1u << u);
          }
        }
        asm volatile("" ::: "memory");
        if (miss && give_up(tries)) {
          stop = 1;
          break;
        }
      }
    };
    const int nslots = (nx + kPoll - 1) / kPoll;
    for (int base = 0; grp + base * a.ngrp < a.P; base += nslot) {
      const int ns =
          kMany ? min((int)nslot, (a.P - 1 - grp) / a.ngrp - base + 1) : 1;
      __syncthreads();  // the last pulses' records have been read
      __syncthreads();  // these are there
      for (int n = 0; n < attempts; ++n) {
        const unsigned act = live_slots(ns);
        if (act == 0) break;
        for (int s = 0; s < kStages; ++s) {
          for (unsigned m = act; m; m &= m - 1) {
            const int b = kMany ? __builtin_ctz(m) : 0;
            const unsigned buf = b * kXbCopies + ((bits2(xcopy, b) + s) & 3u);
            double2 *xs = xs0 + par * nchp * 64;
            if (nslots <= 1) {
              poll(buf, xs, 0, Int<1>());
            } else if (nslots <= 2) {
              poll(buf, xs, 0, Int<2>());
            } else if (nslots <= 4) {
              poll(buf, xs, 0, Int<4>());
            } else {
              // one row first: while it is not there, the others are not
              // asked for
              poll(buf, xs, 0, Int<1>());
              for (int u = 1; u < nslots; u += 8) poll(buf, xs, u, Int<8>());
            }
            __syncthreads();
            if (stop) return;  // uniform over the workgroup
            par ^= 1;
          }
        }
        // ---- step control: every quad's (error max, |y|^2), a wave a slot.
        // k_finalize's order: 256 strided sums (four a lane), then halves of
        // 128, 64 and, across the wave, 32 .. 1
        for (unsigned m = act; m; m &= m - 1) {
          const int b = kMany ? __builtin_ctz(m) : 0;
          if ((b & 3) != w - kRwCompute) continue;
          const int p = grp + (base + b) * a.ngrp;
          double em4[4] = {}, ns4[4] = {};
          bool lost = false;
          for (int i0 = lane; i0 < (int)NQ && !lost; i0 += 256) {
            double2 v[4];
            unsigned miss = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (i0 + u * 64 < (int)NQ) miss |= 1u << u;
            const unsigned r0 = (b * 3 + bits2(rcopy, b)) * NQ + i0;
            for (int tries = 1; miss; ++tries) {
              double2 q[4];
#pragma unroll
              for (int u = 0; u < 4; ++u)
                q[u] = dev_load(rr, (miss >> u) & 1u ? (r0 + u * 64) * 16u
                                                     : kOut);
#pragma unroll
              for (int u = 0; u < 4; ++u)
                if (((miss >> u) & 1u) && !is_unset(q[u].x) &&
                    !is_unset(q[u].y)) {
                  v[u] = q[u];
                  miss &= ~(1u << u);
                }
              asm volatile("" ::: "memory");
              if (miss && give_up(tries)) {
                stop = 1;
                lost = true;
                break;
              }
            }
            if (lost) break;
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (i0 + u * 64 < (int)NQ) {
                em4[u] = v[u].x > em4[u] ? v[u].x : em4[u];
                ns4[u] += v[u].y;
              }
          }
          auto mx = [](double p, double q) { return p > q ? p : q; };
          double em = mx(mx(em4[0], em4[2]), mx(em4[1], em4[3]));
          double n2 = (ns4[0] + ns4[2]) + (ns4[1] + ns4[3]);
#pragma unroll
          for (int o = 32; o > 0; o >>= 1) {
            em = mx(em, __shfl_xor(em, o));
            n2 += __shfl_xor(n2, o);
          }
          if (lane == 0) cl[b] = control_step(cl[b], em, n2, p, a.hs);
          // the record is in LDS before the wave's other lanes read it
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_wave_barrier();
          if (lane < kStages && !cl[b].done)
            cl[b].Fs[lane] =
                stage_field(cl[b], lane, p, a.Ftab, a.pulses, a.env);
        }
        advance(act);
        __syncthreads();
        if (stop) return;
      }
      if (wgi == 0 && tp < ns) a.ctl[grp + (base + tp) * a.ngrp] = cl[tp];
    }
    return;
  }

  // ================= the computing waves =================
  // wave w owns quads w, w + 4, .. of the workgroup, lanes 0, 16, 32, 48
  // their rows
  bool own[kQ];
  int lr[kQ];
  unsigned row[kQ];
  double e[kQ];
#pragma unroll
  for (int m = 0; m < kQ; ++m) {
    lr[m] = (w + m * kRwCompute) * kRwQuad + (lane >> 4);
    own[m] = (lane & 15) == 0 && lr[m] < g.nrows;
    row[m] = (unsigned)(d.off[L] + g.row0 + lr[m]);
    e[m] = 0.0;
    if (own[m]) e[m] = a.E[row[m]];
  }
  // the first quad's first chunks (zeros beyond the last)
  double2 R[kReg + 1][2];
#pragma unroll
  for (int c = 0; c < kReg; ++c)
#pragma unroll
    for (int p = 0; p < 2; ++p)
      R[c][p] = c < nch && w < nq
                    ? D2[((long long)w * nch + c) * 128 + p * 64 + lane]
                    : make_double2(0.0, 0.0);
  // state and stage input of the own rows: with several slots in LDS
  double2 x[kQ], xin[kQ], v[kQ];
  for (int base = 0; grp + base * a.ngrp < a.P; base += nslot) {
    const int ns =
        kMany ? min((int)nslot, (a.P - 1 - grp) / a.ngrp - base + 1) : 1;
    __syncthreads();
    if (t < ns) cl[t] = a.ctl[grp + (base + t) * a.ngrp];
#pragma unroll
    for (int m = 0; m < kQ; ++m)
      if (own[m])
        for (int b = 0; b < ns; ++b) {
          x[m] = a.X[(long long)row[m] * a.P + grp + (base + b) * a.ngrp];
          if (kMany) own_rows[b * slot_n + kStages * nr4 + lr[m]] = x[m];
        }
    __syncthreads();
    for (int n = 0; n < attempts; ++n) {
      const unsigned act = live_slots(ns);
      if (act == 0) break;
      for (unsigned mb = act; mb; mb &= mb - 1) {
        const int b = kMany ? __builtin_ctz(mb) : 0;
        double2 *xv = own_rows + b * slot_n + kStages * nr4;
        const unsigned buf = b * kXbCopies + bits2(xcopy, b);
        const unsigned rc = bits2(rcopy, b);
        const unsigned rnext = b * 3 + (rc == 2 ? 0u : rc + 1);
#pragma unroll
        for (int m = 0; m < kQ; ++m) {
          if (own[m]) {
            if (kMany) x[m] = xv[lr[m]];
            if (kMany) xv[nr4 + lr[m]] = x[m];
            xin[m] = x[m];
            dev_store(rx, (buf * N + row[m]) * 16u, publishable(x[m]));
          }
          // the reduction's copy last read two attempts ago, whose results
          // every workgroup has used since
          if (lane == 0 && own[m])
            dev_store(rr, (rnext * NQ + g.quad0 + w + m * kRwCompute) * 16u,
                      unset);
        }
      }
      for (int s = 0; s < kStages; ++s) {
        const bool last = s == kStages - 1;
        for (unsigned mb = act; mb; mb &= mb - 1) {
          const int b = kMany ? __builtin_ctz(mb) : 0;
          const unsigned c0 = bits2(xcopy, b) + s, bx = b * kXbCopies;
          const unsigned b1 = bx + ((c0 + 1) & 3u), b3 = bx + ((c0 + 3) & 3u);
          double2 *Ks = own_rows + b * slot_n;
          double2 *xv = Ks + kStages * nr4, *xiv = xv + nr4;
          const double2 *xs = xs0 + par * nchp * 64 + lane;
          // while the stage input arrives: the tableau sums of the next one
          // but for k_s (stage_row's terms in stage_row's order)
          const double F = cl[b].Fs[s], h = cl[b].hc;
          const double co = h * coef[s][s];
          double2 err[kQ] = {};
#pragma unroll
          for (int m = 0; m < kQ; ++m) {
            if (!own[m]) continue;
            if (kMany) x[m] = xv[lr[m]];
            if (kMany) xin[m] = xiv[lr[m]];
            v[m] = x[m];
            if (!last) {
#pragma unroll 4
              for (int j = 0; j < s; ++j) {
                const double cj = h * coef[s][j];
                const double2 kj = Ks[j * nr4 + lr[m]];
                v[m].x = fma(cj, kj.x, v[m].x);
                v[m].y = fma(cj, kj.y, v[m].y);
              }
            } else {
#pragma unroll 4
              for (int j = 0; j < kStages - 1; ++j) {
                const double cb = h * coef[kStages - 1][j],
                             cd = h * coef[kStages][j];
                const double2 kj = Ks[j * nr4 + lr[m]];
                v[m].x = fma(cb, kj.x, v[m].x);
                v[m].y = fma(cb, kj.y, v[m].y);
                err[m].x = fma(cd, kj.x, err[m].x);
                err[m].y = fma(cd, kj.y, err[m].y);
              }
            }
          }
          __syncthreads();
          if (stop) return;  // uniform over the workgroup
#pragma unroll
          for (int m = 0; m < kQ; ++m) {
            const int q = w + m * kRwCompute;
            if (q >= nq) continue;  // uniform over the wave
            double2 acc[4] = {};
            // every x is read a group of four chunks ahead (past the last
            // group that is not used; the launch's LDS reaches there)
            double2 xn[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) xn[u] = xs[u * 64];
#pragma unroll
            for (int c0 = 0; c0 < kReg; c0 += 4) {
              if (c0 < nch) {
                double2 xc[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                  xc[u] = xn[u];
                  xn[u] = xs[(c0 + 4 + u) * 64];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                  quad_fma(acc, R[c0 + u][0], R[c0 + u][1], xc[u]);
              }
            }
            int c = kReg;
            const int cl1 = min(c + g.nlds, nch);
            const double2 *Dr = Dl + ((long long)q * g.nlds - c) * 128 + lane;
#pragma unroll 4
            for (; c < cl1; ++c)
              quad_fma(acc, Dr[c * 128], Dr[c * 128 + 64], xs[c * 64]);
            if (c < nch) {
              // the chunks past the LDS share
              const double2 *Dg = D2 + (long long)q * nch * 128 + lane;
#pragma unroll 4
              for (; c < nch; ++c)
                quad_fma(acc, Dg[c * 128], Dg[c * 128 + 64], xs[c * 64]);
            }
            const double2 cs = quad_reduce(acc, lane);
            double errv = 0.0, nrm2 = 0.0;
            if (own[m]) {
              const double2 k =
                  stage_deriv(gauge, e[m], xin[m], F, cs, make_double2(0.0, 0.0));
              if (!last) {
                v[m].x = fma(co, k.x, v[m].x);
                v[m].y = fma(co, k.y, v[m].y);
                // this slot's rows unset a stage ago have landed: two stores
                // a quad and stage, so with other slots in between they are
                // older than the last two
                if (kMany && (act & (act - 1)))
                  asm volatile("s_waitcnt vmcnt(2)" ::: "memory");
                else
                  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                dev_store(rx, (b1 * N + row[m]) * 16u, publishable(v[m]));
                xin[m] = v[m];
                if (kMany) xiv[lr[m]] = v[m];
              } else {
                const double cb = h * cB[kStages - 1], cd = h * cDB[kStages - 1];
                v[m].x = fma(cb, k.x, v[m].x);
                v[m].y = fma(cb, k.y, v[m].y);
                err[m].x = fma(cd, k.x, err[m].x);
                err[m].y = fma(cd, k.y, err[m].y);
                const double2 k1 = Ks[lr[m]];
                const Ctl &c = cl[b];
                const double ex =
                    fabs(err[m].x) / (c.atol + c.rtol * (fabs(x[m].x) + h * fabs(k1.x)));
                const double ey =
                    fabs(err[m].y) / (c.atol + c.rtol * (fabs(x[m].y) + h * fabs(k1.y)));
                errv = ex > ey ? ex : ey;
                nrm2 = abs2(v[m].x, v[m].y);
                if (kMany) xiv[lr[m]] = v[m];
              }
              Ks[s * nr4 + lr[m]] = k;
            }
            if (last) {
              const double2 q2 = quad_norms(errv, nrm2);
              if (lane == 0) en[b][q] = q2;
            }
          }
          // copy b3 (stage g - 1's) has been read by all its readers
#pragma unroll
          for (int m = 0; m < kQ; ++m)
            if (own[m]) dev_store(rx, (b3 * N + row[m]) * 16u, unset);
          par ^= 1;
        }
      }
      // ---- step control
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      for (unsigned mb = act; mb; mb &= mb - 1) {
        const int b = kMany ? __builtin_ctz(mb) : 0;
        const unsigned rc = b * 3 + bits2(rcopy, b);
#pragma unroll
        for (int m = 0; m < kQ; ++m) {
          const int q = w + m * kRwCompute;
          if (lane == 0 && q < nq)
            dev_store(rr, (rc * NQ + g.quad0 + q) * 16u, publishable(en[b][q]));
        }
      }
      __syncthreads();
      if (stop) return;
      for (unsigned mb = act; mb; mb &= mb - 1) {
        const int b = kMany ? __builtin_ctz(mb) : 0;
        const Ctl &c = cl[b];
        if (!c.accept) continue;
        double2 *xv = own_rows + b * slot_n + kStages * nr4;
#pragma unroll
        for (int m = 0; m < kQ; ++m) {
          if (!own[m]) continue;
          if (kMany) v[m] = xv[nr4 + lr[m]];
          x[m] = make_double2(v[m].x / c.nrm, v[m].y / c.nrm);
          if (kMany) xv[lr[m]] = x[m];
          if ((int)row[m] == a.track && c.nlog >= 1 && c.nlog <= a.logcap) {
            LogEnt le;
            le.t = c.t;
            le.h = c.hacc;
            le.pop = abs2(x[m].x, x[m].y);
            a.log[(long long)(c.nlog - 1) * a.P + grp + (base + b) * a.ngrp] =
                le;
          }
        }
      }
      advance(act);
    }
#pragma unroll
    for (int m = 0; m < kQ; ++m)
      if (own[m])
        for (int b = 0; b < ns; ++b)
          a.X[(long long)row[m] * a.P + grp + (base + b) * a.ngrp] =
              kMany ? own_rows[b * slot_n + kStages * nr4 + lr[m]] : x[m];
  }
}

template <int kQ, bool kMany>
__global__ __launch_bounds__(kRwThreads) void k_rows_run(
    typename RowArgs<kMany>::type args) {
  int blk = blockIdx.x;
  if constexpr (kMany) {
    int i = 0;
    for (; i + 1 < args.n; ++i) {
      const int n = args.run[i].nwg * args.run[i].ngrp;
      if (blk < n) break;
      blk -= n;
    }
    rows_run<kQ, kMany>(args.run[i], blk);
  } else {
    rows_run<kQ, kMany>(args, blk);
  }
}

template __global__ void k_rows_run<1, false>(RowRun);
template __global__ void k_rows_run<2, false>(RowRun);
template __global__ void k_rows_run<4, false>(RowRun);
template __global__ void k_rows_run<1, true>(RowRuns);

// ---------------------------------------------------------------------
// Persistent tile kernel: whole attempts of one pulse on a larger system in
// one cooperative launch, one workgroup of eight waves per compute unit.
// The groups (16 rows x 256 columns, 32 KB) of the GEMV store, in the order
// of pair, column block and row, are cut into one equal run per workgroup;
// a group serves both D x_{L+1} and D^T x_L, so every dipole is read once a
// stage.  The first kTlReg groups of a run stay in registers and as many as
// fit in LDS for the whole launch; the others are streamed through a ring of
// kTlRing groups in registers, in alternating direction from stage to stage,
// so that the last ones of a stage are found in L2 by the next.
//
// A stage: the stage input of the run's rows and columns is polled into LDS;
// per group, a lane's eight products go to the row sum (reduced over the 16
// column lanes of a wave's row at once, over the waves every eight groups)
// and to the column accumulators (kept for a segment, reduced over the 16
// row lanes at its end); the partials are published; the workgroup that owns
// a row polls its partials (one per column block of D, one per segment of
// D^T), sums them in a fixed order, runs the stage algebra and publishes the
// next stage input.  Two exchanges a stage, each the same sentinel scheme as
// above: three copies of the inputs xb, of the partials pb (a slot is unset
// one stage after its readers have passed it) and of the step control's
// per-workgroup maxima rb.
//
// What bounds it: up to about 60 MB, where nothing or little is streamed,
// the two exchanges and the polls (about 8 us a stage); past that the
// streamed bytes, at 5.3 to 5.7 TB/s of the 6.9 TB/s that long reads reach
// over the whole stage (the copies in registers and LDS, 50 to 59 MB over the
// device, are not read again; the fill and drain of the ring and the exchanges
// are the rest).  4000 x 4: 50.3 of 393.2 MB kept, 323 MB a stage fetched past
// L2 by the counters.
// Per attempt, against launches of k_gemv_tile and k_stage1: blocks 1500 x 4
// (54 MB) 225 -> 127 us, 2000 x 4 (96 MB) 306 -> 181 us, blocks 2200, 2600,
// 1800, 2400, 2000 355 against 482 us, 998 x 21 (159 MB) 473 -> 312 us,
// 4000 x 4 (384 MB) 925 -> 763 us, 6000 x 3 (576 MB) 1406 -> 1278 us.
// Tried, and no faster: a ring of three, one to three groups in registers,
// the columns' stage input in registers instead of LDS, runs weighted by
// the columns they read.
// ---------------------------------------------------------------------
// Sixteen values summed over the 16 lanes of a row: lane i returns value i
// (bit 3 .. 0 of the index taken by row_ror:8, row_half_mirror and the two
// quad swaps in turn).
__device__ __forceinline__ double sum16_transposed(const double (&v)[16],
                                                   int tr) {
  const bool b3 = (tr & 8) != 0, b2 = (tr & 4) != 0, b1 = (tr & 2) != 0,
             b0 = (tr & 1) != 0;
  double p[8], q[4], r[2];
#pragma unroll
  for (int m = 0; m < 8; ++m)
    p[m] = (b3 ? v[8 + m] : v[m]) + dpp_perm<0x128>(b3 ? v[m] : v[8 + m]);
#pragma unroll
  for (int m = 0; m < 4; ++m)
    q[m] = (b2 ? p[4 + m] : p[m]) + dpp_perm<0x141>(b2 ? p[m] : p[4 + m]);
#pragma unroll
  for (int m = 0; m < 2; ++m)
    r[m] = (b1 ? q[2 + m] : q[m]) + dpp_perm<0x4E>(b1 ? q[m] : q[2 + m]);
  return (b0 ? r[1] : r[0]) + dpp_perm<0xB1>(b0 ? r[0] : r[1]);
}

__global__ __launch_bounds__(kGvThreads) void k_tiles_run(
    TileRun a, const SysDesc *__restrict__ dp,
    const TileDesc *__restrict__ tdp) {
  typedef double dv2 __attribute__((ext_vector_type(2)));
  const SysDesc &d = *dp;
  const TileDesc &td = *tdp;
  const TileWg g = a.wg[blockIdx.x];
  const TileSeg *__restrict__ segs = a.seg + g.seg0;
  const int t = threadIdx.x, lane = t & 63;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int tr = t & 15, cg = t >> 4;
  constexpr int kWv = kGvThreads / 64;
  const int gauge = d.gauge, ngroups = g.ngroups;
  const int attempts = g.quit > 0 ? g.quit - 1 : a.attempts;
  const int nown = g.nrows;
  const int nitems = g.nrs + g.ncs;

  // LDS: the stage input over the workgroup's row groups and over its
  // segments' columns, the waves' row sums of up to eight groups (two
  // copies), the gathered partials and the 13 stage derivatives of its own
  // rows, the resident groups
  extern __shared__ __align__(16) unsigned char smem[];
  double2 *xrow = reinterpret_cast<double2 *>(smem);
  double2 *xcol = xrow + a.xs_rows;
  double2 *rowbuf = xcol + a.xs_segs * kGvTC;        // [2][kWv][kGvTR]
  double2 *pbuf = rowbuf + 2 * kWv * kGvTR;          // [wave][row]
  double2 *Ks = pbuf + kWv * nown;                   // [stage][row]
  // group q: its index in the store, its rows and columns inside the block
  int4 *gtab = reinterpret_cast<int4 *>(Ks + kStages * nown);
  // piece i of the stage input: first row, LDS place, rows inside the block
  int4 *ptab = gtab + ngroups;
  // segment: groups, first group, rows and columns of the block below its
  // first; where its row and column partials start
  int4 *stab = ptab + a.xs_pieces;
  dv2 *Dl = reinterpret_cast<dv2 *>(stab + 2 * a.xs_segs);
  __shared__ Ctl cl;
  __shared__ double se[256], sn[256];
  __shared__ double coef[kStages + 1][kStages];
  __shared__ int stop;
  __shared__ int nslot[kTlMaxRows];

  const unsigned N = (unsigned)a.N, PN = (unsigned)td.part_n,
                 NW = (unsigned)a.nwg;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.xb, (short)0, (int)(3u * N * 16u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.pb, (short)0, (int)(3u * PN * 16u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.rb, (short)0, (int)(3u * NW * 16u), 0x00020000);
  constexpr unsigned kOut = 0x80000000u;  // beyond any buffer range
  const double u_ = __longlong_as_double((long long)kUnset);
  const double2 unset = make_double2(u_, u_);

  // this lane's four column pairs of group q (a lane beyond the block
  // re-reads its first pair, a cache hit, and meets zeros)
  const dv2 *Dt = reinterpret_cast<const dv2 *>(a.Dg) + t;
  auto load_group = [&](int q, dv2 (&v)[kGvColPairIter]) {
    const int4 gt = gtab[q];
    const int job = __builtin_amdgcn_readfirstlane(gt.x);
    const int nc = __builtin_amdgcn_readfirstlane(gt.z);
    const dv2 *base = Dt + (long long)job * (kGvColPairIter * kGvThreads);
    const bool rv = tr < __builtin_amdgcn_readfirstlane(gt.y);
#pragma unroll
    for (int j = 0; j < kGvColPairIter; ++j) {
      const bool cv = 2 * (cg + 32 * j) < nc;
      int o = (rv && cv) ? j * kGvThreads : 0;
      asm volatile("" : "+v"(o));
      v[j] = base[o];
    }
  };

  if (t == 0) {
    cl = a.ctl[0];
    stop = 0;
    if (a.limit_ms < 0) {  // no wait at all
      stop = 1;
      __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    } else if (a.start_ms > 0 &&
               !all_started(a.arrived, a.abort_flag, a.start_ms)) {
      stop = 1;
    }
  }
  if (t < (kStages + 1) * kStages) {
    const int s = t / kStages, j = t - s * kStages;
    coef[s][j] = s < kStages - 1 ? cA[s + 1][j] : s == kStages - 1 ? cB[j] : cDB[j];
  }
  // the tables of the groups and of the stage input's pieces (64 rows each:
  // a segment's rows, then its 256 columns)
  int npiece = 0;
  {
    int q0 = 0;
    for (int s = 0; s < g.nseg; ++s) {
      const TileSeg sg = segs[s];
      const int sL = d.off[sg.L + 1] - d.off[sg.L];
      const int sL1 = d.off[sg.L + 2] - d.off[sg.L + 1];
      const int nr = (sg.ng + 3) / 4;
      for (int k = t; k < sg.ng; k += kGvThreads) {
        const int gi = sg.g0 + k, rb = gi >> 3;
        const int job = sg.job0 + rb * sg.ncb + (sg.cb + sg.ncb - rb % sg.ncb) % sg.ncb;
        gtab[q0 + k] = make_int4((gi & 7) * a.njobs + job, sL - gi * 16,
                                 sL1 - sg.cb * kGvTC, 0);
      }
      for (int k = t; k < nr + 4; k += kGvThreads) {
        const bool rows = k < nr;
        const int first = rows ? sg.g0 * 16 + k * 64
                               : sg.cb * kGvTC + (k - nr) * 64;
        const int end = rows ? min(sL, (sg.g0 + sg.ng) * 16) : sL1;
        ptab[npiece + k] =
            make_int4(d.off[rows ? sg.L : sg.L + 1] + first,
                      rows ? q0 * 16 + k * 64
                           : a.xs_rows + s * kGvTC + (k - nr) * 64,
                      end - first, rows ? (sg.ng * 16 - k * 64) : 64);
      }
      if (t == 0) {
        stab[2 * s] = make_int4(sg.ng, sg.g0, sL, sL1 - sg.cb * kGvTC);
        stab[2 * s + 1] =
            make_int4(td.rp_off[sg.L] + sg.cb * sL,
                      td.cp_off[sg.L] + sg.slot * sL1 + sg.cb * kGvTC, 0, 0);
      }
      q0 += sg.ng;
      npiece += nr + 4;
    }
  }
  __syncthreads();
  // resident groups: the first kTlReg in registers, the next nlds in LDS
  dv2 R[kTlReg][kGvColPairIter];
#pragma unroll
  for (int q = 0; q < kTlReg; ++q) {
#pragma unroll
    for (int j = 0; j < kGvColPairIter; ++j) R[q][j] = dv2{0.0, 0.0};
    if (q < ngroups) load_group(q, R[q]);
  }
  for (int q = 0; q < g.nlds; ++q) {
    dv2 v[kGvColPairIter];
    load_group(kTlReg + q, v);
#pragma unroll
    for (int j = 0; j < kGvColPairIter; ++j)
      Dl[(q * kGvColPairIter + j) * kGvThreads + t] = v[j];
  }
  // resident groups; at least kTlRing are streamed, or none
  const int nres = ngroups <= kTlReg + g.nlds ? ngroups
                                              : min(kTlReg + g.nlds, ngroups - kTlRing);
  const bool own = t < nown;
  const unsigned row = (unsigned)(d.off[g.L] + g.row0 + t);
  double2 x = make_double2(0.0, 0.0);
  double e = 0.0;
  if (own) {
    x = a.X[row];
    e = a.E[row];
  }
  // D^T x_{L-1} partials of each own row
  if (own)
    nslot[t] = g.ncs > 0
                   ? a.nslot[td.cs_off[g.L - 1] + (g.row0 + t) / kGvTC]
                   : 0;
  const int cp0 = g.ncs > 0 ? td.cp_off[g.L - 1] + g.row0 : 0;
  const int rp0 = g.nrs > 0 ? td.rp_off[g.L] + g.row0 : 0;
  const int sOwn = d.off[g.L + 1] - d.off[g.L];
  __syncthreads();
  if (stop) return;  // uniform

  long long t_wait = 0;
  auto give_up = [&](int tries) -> bool {
    if ((tries & 63) != 0) return false;
    const long long now = wall_clock64();
    if (tries == 64) t_wait = now;
    const bool late = now - t_wait > (long long)a.limit_ms * 100000;
    if (late)
      __hip_atomic_store(a.abort_flag, 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    return late || __hip_atomic_load(a.abort_flag, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT) != 0;
  };
  // polls U values per lane (off[u] in 16 bytes, ~0u: none) until all are set
  auto poll = [&](__amdgpu_buffer_rsrc_t r, auto width, unsigned *off,
                  double2 *v) {
    constexpr int U = decltype(width)::value;
    unsigned miss = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (off[u] != ~0u) miss |= 1u << u;
      v[u] = make_double2(0.0, 0.0);
    }
    for (int tries = 1; __any(miss != 0); ++tries) {
      double2 q[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        q[u] = dev_load(r, (miss >> u) & 1u ? off[u] * 16u : kOut);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (((miss >> u) & 1u) && !is_unset(q[u].x) && !is_unset(q[u].y)) {
          v[u] = q[u];
          miss &= ~(1u << u);
        }
      asm volatile("" ::: "memory");
      if (miss && give_up(tries)) {
        stop = 1;
        break;
      }
    }
  };

  unsigned buf = 0, rbuf = 0;  // exchange copies of the coming stage, reduction
  // streamed groups: kTlRing in flight, in turn
  const int nstr = ngroups - nres;
  // the k-th streamed group of a sweep in direction rev; past the sweep's
  // end, the next stage's sweep (which starts where this one ends, but for
  // the step from the last stage to the first).  With fewer streamed groups
  // than the ring holds, all of them are resident instead (see nres).
  auto streamed = [&](int k, int rev, int rev_next) {
    if (k >= nstr) {
      k -= nstr;
      rev = rev_next;
    }
    return rev ? ngroups - 1 - k : nres + k;
  };
  dv2 S[kTlRing][kGvColPairIter];
#pragma unroll
  for (int m = 0; m < kTlRing; ++m) {
#pragma unroll
    for (int j = 0; j < kGvColPairIter; ++j) S[m][j] = dv2{0.0, 0.0};
    if (nstr > 0) load_group(streamed(m, 0, 1), S[m]);
  }
  int ph = 0;  // which of them comes next
  for (int n = 0; n < attempts && !cl.done; ++n) {
    const double h = cl.hc;
    const unsigned rnext = rbuf == 2 ? 0 : rbuf + 1;
    double2 xin = x, v = x;
    double errv = 0.0, nrm2 = 0.0;
    if (own) dev_store(rx, (buf * N + row) * 16u, publishable(x));
    if (t == 0) dev_store(rr, (rnext * NW + blockIdx.x) * 16u, unset);
    for (int s = 0; s < kStages; ++s) {
      const unsigned b1 = buf == 2 ? 0 : buf + 1, b2 = b1 == 2 ? 0 : b1 + 1;
      const int rev = s & 1;
      const bool last = s == kStages - 1;
      // ---- while the stage input arrives: the tableau sums of the next one
      // but for k_s (stage_row's terms in stage_row's order)
      double2 err = make_double2(0.0, 0.0);
      if (own) {
        v = x;
        if (!last) {
#pragma unroll 4
          for (int j = 0; j < s; ++j) {
            const double cj = h * coef[s][j];
            const double2 kj = Ks[j * nown + t];
            v.x = fma(cj, kj.x, v.x);
            v.y = fma(cj, kj.y, v.y);
          }
        } else {
#pragma unroll 4
          for (int j = 0; j < kStages - 1; ++j) {
            const double cb = h * coef[kStages - 1][j], cd = h * coef[kStages][j];
            const double2 kj = Ks[j * nown + t];
            v.x = fma(cb, kj.x, v.x);
            v.y = fma(cb, kj.y, v.y);
            err.x = fma(cd, kj.x, err.x);
            err.y = fma(cd, kj.y, err.y);
          }
        }
      }
      // ---- the stage input (the owners' waves fetch last)
      for (int i = kWv - 1 - w; i < npiece; i += 3 * kWv) {
        unsigned off[3];
        int at[3];
        double2 val[3];
#pragma unroll
        for (int u = 0; u < 3; ++u) {
          off[u] = ~0u;
          at[u] = -1;
          if (i + u * kWv < npiece) {
            const int4 pt = ptab[i + u * kWv];
            if (lane < pt.w) at[u] = pt.y + lane;
            if (lane < min(pt.z, pt.w)) off[u] = buf * N + pt.x + lane;
          }
        }
        poll(rx, Int<3>(), off, val);
#pragma unroll
        for (int u = 0; u < 3; ++u)
          if (at[u] >= 0) xrow[at[u]] = val[u];
      }
      // partials unset in the last sweep have landed: in this one another
      // wave may write their slots
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (stop) return;  // uniform over the workgroup
      // ---- the coupling sums, segment by segment
      int q = rev ? ngroups - 1 : 0;  // group within the workgroup
      int flush = 0;                  // row-sum batches of this stage
      for (int si = 0; si < g.nseg; ++si) {
        const int sx = rev ? g.nseg - 1 - si : si;
        const int4 st0 = stab[2 * sx], st1 = stab[2 * sx + 1];
        const int s_ng = __builtin_amdgcn_readfirstlane(st0.x);
        const int s_g0 = __builtin_amdgcn_readfirstlane(st0.y);
        const int s_rows = __builtin_amdgcn_readfirstlane(st0.z);
        const int s_cols = __builtin_amdgcn_readfirstlane(st0.w);
        const int s_rp = __builtin_amdgcn_readfirstlane(st1.x);
        const int s_cp = __builtin_amdgcn_readfirstlane(st1.y);
        const double2 *xc = xcol + sx * kGvTC + 2 * cg;
        double2 acc[kGvColPairIter][2] = {};
        int nb = 0;  // groups in the row-sum batch
        auto consume = [&](const dv2 (&cur)[kGvColPairIter]) {
          const double2 xr = xrow[q * 16 + tr];
          double pre = 0.0, pim = 0.0;
#pragma unroll
          for (int j = 0; j < kGvColPairIter; ++j) {
            const dv2 dv = cur[j];
            const double2 xa = xc[64 * j], xb = xc[64 * j + 1];
            pre = fma(dv.x, xa.x, pre);
            pim = fma(dv.x, xa.y, pim);
            pre = fma(dv.y, xb.x, pre);
            pim = fma(dv.y, xb.y, pim);
            acc[j][0].x = fma(dv.x, xr.x, acc[j][0].x);
            acc[j][0].y = fma(dv.x, xr.y, acc[j][0].y);
            acc[j][1].x = fma(dv.y, xr.x, acc[j][1].x);
            acc[j][1].y = fma(dv.y, xr.y, acc[j][1].y);
          }
          // the row sums over the wave's four column groups: the lower wave
          // half ends with the real part
          const double ps = add_xor16(pair_sum<true>(pre, pim));
          if ((lane & 16) == 0)
            reinterpret_cast<double *>(
                rowbuf + ((flush & 1) * kWv + w) * kGvTR + nb * 16 +
                tr)[lane >> 5] = ps;
        };
        for (int k = 0; k < s_ng; ++k) {
          if (q < min(kTlReg, nres)) {
#pragma unroll
            for (int m = 0; m < kTlReg; ++m)
              if (q == m) consume(R[m]);
          } else if (q < nres) {
            dv2 cur[kGvColPairIter];
#pragma unroll
            for (int j = 0; j < kGvColPairIter; ++j)
              cur[j] = Dl[((q - kTlReg) * kGvColPairIter + j) * kGvThreads + t];
            consume(cur);
          } else {
            const int qn = streamed(
                (rev ? ngroups - 1 - q : q - nres) + kTlRing, rev,
                last ? 0 : !rev);
#pragma unroll
            for (int m = 0; m < kTlRing; ++m)
              if (ph == m) {
                consume(S[m]);
                load_group(qn, S[m]);
              }
            ph = ph == kTlRing - 1 ? 0 : ph + 1;
          }
          ++nb;
          if (nb == 8 || k == s_ng - 1) {
            // flush: sum over the 8 waves in a fixed order
            __syncthreads();
            const int r = t >> 1, comp = t & 1;
            if (r < nb * 16) {
              const double *b = reinterpret_cast<const double *>(
                  rowbuf + (flush & 1) * kWv * kGvTR + r) + comp;
              double sum = 0.0;
#pragma unroll
              for (int ww = 0; ww < kWv; ++ww) sum += b[ww * 2 * kGvTR];
              // batch slot r / 16 back to the group
              const int kk = rev ? s_ng - 1 - (k - (nb - 1 - (r >> 4)))
                                 : k - (nb - 1 - (r >> 4));
              const int gr = (s_g0 + kk) * 16 + (r & 15);
              if (gr < s_rows) {
                const unsigned slot = (unsigned)(s_rp + gr);
                dev_store1(rp, (buf * PN + slot) * 16u + comp * 8u,
                           publishable1(sum));
                dev_store1(rp, (b2 * PN + slot) * 16u + comp * 8u, u_);
              }
            }
            nb = 0;
            ++flush;
          }
          q += rev ? -1 : 1;
        }
        // the segment's column sums over the 16 row lanes
        double vals[16];
#pragma unroll
        for (int j = 0; j < kGvColPairIter; ++j)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            vals[(j * 2 + c) * 2] = acc[j][c].x;
            vals[(j * 2 + c) * 2 + 1] = acc[j][c].y;
          }
        const double cv = sum16_transposed(vals, tr);
        const double co = dpp_perm<0xB1>(cv);  // the other part
        const int cidx = tr >> 1;
        const int col = 2 * (cg + 32 * (cidx >> 1)) + (cidx & 1);
        if ((tr & 1) == 0 && col < s_cols) {
          const unsigned slot = (unsigned)(s_cp + col);
          dev_store(rp, (buf * PN + slot) * 16u,
                    publishable(make_double2(cv, co)));
          dev_store(rp, (b2 * PN + slot) * 16u, unset);
        }
      }
      // ---- the own rows: gather the partials, wave w the items w, w + 8, ..
      // (D x_{L+1} with the sign of the gauge's formula)
#pragma unroll
      for (int hf = 0; hf < kTlMaxRows / 64; ++hf) {
        const int r = hf * 64 + lane;
        if (hf * 64 >= nown) break;
        double2 sum = make_double2(0.0, 0.0);
        for (int i = w; i < nitems; i += 3 * kWv) {
          unsigned off[3];
          double2 val[3];
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            const int it = i + u * kWv;
            off[u] = ~0u;
            if (it < nitems && r < nown) {
              if (it >= g.ncs)
                off[u] = buf * PN + rp0 + (it - g.ncs) * sOwn + r;
              else if (it < nslot[r])
                off[u] = buf * PN + cp0 + it * sOwn + r;
            }
          }
          poll(rp, Int<3>(), off, val);
#pragma unroll
          for (int u = 0; u < 3; ++u) {
            const bool neg = gauge == 0 && i + u * kWv >= g.ncs;
            sum.x += neg ? -val[u].x : val[u].x;
            sum.y += neg ? -val[u].y : val[u].y;
          }
        }
        if (r < nown) pbuf[w * nown + r] = sum;
      }
      __syncthreads();
      if (stop) return;  // uniform over the workgroup
      if (own) {
        double2 cs = make_double2(0.0, 0.0);
#pragma unroll
        for (int k = 0; k < kWv; ++k) {
          const double2 p = pbuf[k * nown + t];
          cs.x += p.x;
          cs.y += p.y;
        }
        const double2 k = stage_deriv(gauge, e, xin, cl.Fs[s], cs,
                                      make_double2(0.0, 0.0));
        const double co = h * coef[s][s];
        if (!last) {
          v.x = fma(co, k.x, v.x);
          v.y = fma(co, k.y, v.y);
          xin = v;
          // the rows unset a stage ago have landed
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          dev_store(rx, (b1 * N + row) * 16u, publishable(v));
        } else {
          const double cd = h * coef[kStages][kStages - 1];
          v.x = fma(co, k.x, v.x);
          v.y = fma(co, k.y, v.y);
          err.x = fma(cd, k.x, err.x);
          err.y = fma(cd, k.y, err.y);
          const double2 k1 = Ks[t];
          const double ex = fabs(err.x) / (cl.atol + cl.rtol * (fabs(x.x) +
                                                                h * fabs(k1.x)));
          const double ey = fabs(err.y) / (cl.atol + cl.rtol * (fabs(x.y) +
                                                                h * fabs(k1.y)));
          errv = ex > ey ? ex : ey;
          nrm2 = abs2(v.x, v.y);
        }
        Ks[s * nown + t] = k;
        // every reader of this stage's input has given its partials
        dev_store(rx, (buf * N + row) * 16u, unset);
      }
      buf = b1;
    }
    // ---- step control: the workgroup's rows, then all workgroups
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (t < 256) {
      se[t] = errv;
      sn[t] = nrm2;
    }
    __syncthreads();
    auto mx = [](double p, double q) { return p > q ? p : q; };
    if (w == 0) {
      double em = mx(mx(se[t], se[t + 128]), mx(se[t + 64], se[t + 192]));
      double ns = (sn[t] + sn[t + 128]) + (sn[t + 64] + sn[t + 192]);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        em = mx(em, __shfl_xor(em, o));
        ns += __shfl_xor(ns, o);
      }
      if (t == 0)
        dev_store(rr, (rbuf * NW + blockIdx.x) * 16u,
                  publishable(make_double2(em, ns)));
    }
    __syncthreads();
    if (t < 256) {
      unsigned off[1] = {t < a.nwg ? rbuf * NW + t : ~0u};
      double2 val[1];
      poll(rr, Int<1>(), off, val);
      se[t] = val[0].x;
      sn[t] = val[0].y;
    }
    __syncthreads();
    if (stop) return;  // uniform over the workgroup
    if (w == 0) {
      double em = mx(mx(se[t], se[t + 128]), mx(se[t + 64], se[t + 192]));
      double ns = (sn[t] + sn[t + 128]) + (sn[t + 64] + sn[t + 192]);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        em = mx(em, __shfl_xor(em, o));
        ns += __shfl_xor(ns, o);
      }
      if (t == 0) cl = control_step(cl, em, ns, 0, a.hs);
      // the record is in LDS before the wave's other lanes read it
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_wave_barrier();
      if (t < kStages && !cl.done)
        cl.Fs[t] = stage_field(cl, t, 0, a.Ftab, a.pulses, a.env);
    }
    rbuf = rnext;
    __syncthreads();
    if (own && cl.accept) {
      x = make_double2(v.x / cl.nrm, v.y / cl.nrm);
      if ((int)row == a.track && cl.nlog >= 1 && cl.nlog <= a.logcap) {
        LogEnt le;
        le.t = cl.t;
        le.h = cl.hacc;
        le.pop = abs2(x.x, x.y);
        a.log[cl.nlog - 1] = le;
      }
    }
  }
  if (own) a.X[row] = x;
  if (blockIdx.x == 0 && t == 0) a.ctl[0] = cl;
}


}  // namespace mpci
