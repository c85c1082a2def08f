// Time-chunk kernels of the fused path (gfx950): the gate outputs' first
// tails, the per-chunk SAIF accumulation, and the SAIF of the resident stimulus
// (the stimulus cut and the tails carried from chunk to chunk are with the
// level kernels, whose scans they share).
//
// A simulation runs as time chunks [F_k, F_k+1) (device.h, ChunkWin).  The
// stimulus stays resident for the whole run as 64-bit words
// (absolute time << 2 | value); each chunk cuts every signal's range
// [lb_k, F_k+1) out of it, in the chunk's relative time, behind a state entry
// (the value before lb_k, X when there is none: src/simulate.cpp:1459-1506
// reads X before a net's first entry).  Gate outputs of chunk k are final
// below F_k+1 (a candidate made at time t has output time >= t, so events at
// or after F_k+1 cannot pre-empt them); their tails (the state entry before
// lb_k+1 and the entries at or after it) seed chunk k+1.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device.h"

namespace gls {

// Chunk 0: every gate output's tail is one X state entry (word 1 at
// relative time 0), tail of gate g at tails[g].
__global__ void k_tails_init(const GateRec* __restrict__ gates, uint32_t ng,
                             uint32_t* __restrict__ tail_len, uint64_t* __restrict__ tail_off,
                             uint32_t* __restrict__ tails) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ng) return;
  const uint32_t net = gates[g].out_net;
  tail_len[net] = 1;
  tail_off[net] = g;
  tails[g] = 1u;
}

// End of chunk k, per gate output: SAIF durations and toggles of the chunk
// join the run's totals, and the net's new entries (after its tail) are
// added to its waveform length.
__global__ void k_saif_accum(const GateRec* __restrict__ gates, uint32_t ng,
                             const unsigned long long* __restrict__ chunk,
                             unsigned long long* __restrict__ saif, const uint32_t* __restrict__ wlen,
                             const uint32_t* __restrict__ tail_len, unsigned long long* __restrict__ wtot,
                             const uint64_t* __restrict__ scal) {
  if (scal[S_TRIP]) return;
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= ng) return;
  const uint32_t net = gates[g].out_net;
  const unsigned long long* c = chunk + (uint64_t)kSaifWords * net;
  unsigned long long* d = saif + (uint64_t)kSaifWords * net;
  d[0] += c[0];
  d[1] += c[1];
  d[2] += c[2];
  d[3] += c[3];
  wtot[net] += wlen[net] - tail_len[net];
}

// SAIF of the resident stimulus signals over the whole window (once per
// run; they are never re-computed per chunk): one block per signal, the net is X before its first entry, an entry holds until the next one (the
// last until the window end), src/simulate.cpp:102-163.
__device__ __forceinline__ void saif_add64(unsigned long long* acc, uint32_t v, uint64_t a,
                                           uint64_t b, uint64_t start, uint64_t end) {
  const uint64_t lo = a > start ? a : start, hi = b < end ? b : end;
  if (hi <= lo) return;
  const uint64_t len = hi - lo;
  if (v == 0) acc[0] += len;
  else if (v == 3) acc[1] += len;
  else acc[2] += len;
}

// (One wavefront per signal waited for its loads 31 times over 2,000 events: 25
// us, three of a hundred of a run of 2,000 cells.)
__global__ __launch_bounds__(256) void k_saif_stim(
    const uint64_t* __restrict__ store, const uint64_t* __restrict__ soff,
    const uint32_t* __restrict__ slen, const uint32_t* __restrict__ snet,
    const uint32_t* __restrict__ sjob, unsigned long long* __restrict__ saif,
    const unsigned long long* __restrict__ win, unsigned long long* __restrict__ wtot) {
  __shared__ unsigned long long s_acc[4][4];
  const uint32_t s = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const uint64_t start = win[2 * sjob[s]], end = win[2 * sjob[s] + 1];
  const uint64_t* w = store + soff[s];
  const uint32_t n = slen[s];
  unsigned long long acc[4] = {0, 0, 0, 0};
  if (threadIdx.x == 0) saif_add64(acc, 1u, 0, n ? (w[0] >> 2) : end, start, end);
  constexpr uint32_t kAhead = 4;  // rounds whose loads are in flight together
  for (uint64_t q0 = threadIdx.x; q0 < n; q0 += 256 * kAhead) {
    uint64_t p[kAhead], e[kAhead], x[kAhead];
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) {
      const uint64_t q = q0 + 256 * i;
      e[i] = q < n ? w[q] : 0;
      p[i] = q < n && q > 0 ? w[q - 1] : 0;
      x[i] = q + 1 < n ? w[q + 1] : 0;
    }
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) {
      const uint64_t q = q0 + 256 * i;
      if (q >= n) break;
      const uint64_t t = e[i] >> 2;
      const uint64_t tn = q + 1 < n ? (x[i] >> 2) : (end > t ? end : t);
      saif_add64(acc, (uint32_t)(e[i] & 3u), t, tn, start, end);
      // stimulus waveforms may repeat a value (scalars are not de-duplicated)
      if (q > 0 && is_toggle((uint32_t)(p[i] & 3u), (uint32_t)(e[i] & 3u)) && t > start && t <= end)
        ++acc[3];
    }
  }
  for (int k = 0; k < 4; ++k) {
    for (int o = 32; o > 0; o >>= 1) acc[k] += __shfl_down(acc[k], o, 64);
    if (lane == 0) s_acc[wid][k] = acc[k];
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    const uint32_t k = threadIdx.x;
    saif[(uint64_t)kSaifWords * snet[s] + k] = s_acc[0][k] + s_acc[1][k] + s_acc[2][k] + s_acc[3][k];
  }
  if (threadIdx.x == 0) wtot[snet[s]] = n;
}

static inline unsigned nblk(uint64_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_tails_init(const GateRec* gates, uint32_t ng, uint32_t* tail_len,
                             uint64_t* tail_off, uint32_t* tails, hipStream_t st) {
  if (ng == 0) return hipSuccess;
  k_tails_init<<<nblk(ng, 256), 256, 0, st>>>(gates, ng, tail_len, tail_off, tails);
  return hipGetLastError();
}

hipError_t launch_saif_accum(const GateRec* gates, uint32_t ng, const unsigned long long* chunk,
                             unsigned long long* saif, const uint32_t* wlen,
                             const uint32_t* tail_len, unsigned long long* wtot, const uint64_t* scal,
                             hipStream_t st) {
  if (ng == 0) return hipSuccess;
  k_saif_accum<<<nblk(ng, 256), 256, 0, st>>>(gates, ng, chunk, saif, wlen, tail_len, wtot, scal);
  return hipGetLastError();
}

// dst[i] += src[i]: a chunk's per-instance gate events join the run's.
__global__ void k_add_u64(unsigned long long* dst, const unsigned long long* src, uint64_t n,
                          const uint64_t* scal) {
  if (scal[S_TRIP]) return;
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] += src[i];
}

hipError_t launch_add_u64(unsigned long long* dst, const unsigned long long* src, uint64_t n,
                          const uint64_t* scal, hipStream_t st) {
  if (n == 0) return hipSuccess;
  k_add_u64<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(dst, src, n, scal);
  return hipGetLastError();
}

hipError_t launch_saif_stim(const uint64_t* store, const uint64_t* soff, const uint32_t* slen,
                            const uint32_t* snet, const uint32_t* sjob, uint32_t ns,
                            unsigned long long* saif, const unsigned long long* win,
                            unsigned long long* wtot, hipStream_t st) {
  if (ns == 0) return hipSuccess;
  k_saif_stim<<<ns, 256, 0, st>>>(store, soff, slen, snet, sjob, saif, win, wtot);
  return hipGetLastError();
}

}  // namespace gls
