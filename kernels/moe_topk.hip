// What surrounds the expert products of a softmax-routed mixture: router product and
// choice, grouping of the token-expert pairs, and the weighted sum of the results.
//
// These took some 20 launches of tensor ops a layer (product, softmax, selection, sort,
// histogram, prefix, gathers, scatter-add): all of them latency at decode sizes, and
// several passes over [T k, H] at prompt sizes.  Three launches instead; the expert
// product reads its rows through the list made here, so the gathered copy is gone, and
// the sum is taken in f32 and rounded once.

#include "common.h"

namespace {

constexpr int kMaxExperts = 64;
constexpr int kMaxTop = 8;

// Eight values of every lane summed over the wave, each in the order of wave_reduce_sum: at every
// step half of them go to half of the lanes, 10 exchanges instead of 48.  Lane l has value l / 8.
DEVINLINE float sums_of_wave(float (&v)[8]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    const int half = 4 >> s, mask = 32 >> s;
    const bool up = lane & mask;
#pragma unroll
    for (int i = 0; i < half; ++i) {
      const float send = up ? v[i] : v[i + half], keep = up ? v[i + half] : v[i];
      v[i] = keep + __shfl_xor(send, mask, 64);
    }
  }
#pragma unroll
  for (int mask = 4; mask >= 1; mask >>= 1) v[0] += __shfl_xor(v[0], mask, 64);
  return v[0];
}

// ids, weights [T, top]: the top largest x[t]·gate[e] and their softmax among themselves.
// The four waves cut K; a workgroup's tokens share what it reads of the gate matrix.
// Bound by the latency of a few dependent loads at decode sizes, by x and the gate
// matrix from L2 at prompt sizes.
template <int kTokens>   // of a workgroup
__global__ __launch_bounds__(256) void moe_topk_kernel(
    int* __restrict__ ids, float* __restrict__ weights,
    const __hip_bfloat16* __restrict__ x,     // [T, K]
    const __hip_bfloat16* __restrict__ gate,  // [E, K]
    const int T, const int E, const int K, const int top) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t0 = blockIdx.x * kTokens;
  __shared__ float part[4][kTokens][8];
  __shared__ float logits[kTokens][kMaxExperts];

  const int per = ((K / 8 + 3) / 4) * 8;      // inputs of a wave, in runs of 8
  const int lo = wave * per, hi = min(lo + per, K);
  for (int e0 = 0; e0 < E; e0 += 8) {
    float acc[kTokens * 8];
#pragma unroll
    for (int i = 0; i < kTokens * 8; ++i) acc[i] = 0.f;
    for (int k = lo + lane * 8; k < hi; k += 512) {
      Vec16<__hip_bfloat16> xv[kTokens], gv[8];
#pragma unroll
      for (int t = 0; t < kTokens; ++t) xv[t] = load16(x + (long)min(t0 + t, T - 1) * K + k);
#pragma unroll
      for (int e = 0; e < 8; ++e) gv[e] = load16(gate + (long)min(e0 + e, E - 1) * K + k);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float xf[kTokens];
#pragma unroll
        for (int t = 0; t < kTokens; ++t) xf[t] = __bfloat162float(xv[t].data[j]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float g = __bfloat162float(gv[e].data[j]);
#pragma unroll
          for (int t = 0; t < kTokens; ++t) acc[t * 8 + e] = __builtin_fmaf(xf[t], g, acc[t * 8 + e]);
        }
      }
    }
    if constexpr (kTokens == 1) {
      const float v = sums_of_wave(acc);
      if (lane % 8 == 0) part[wave][0][lane / 8] = v;
    } else {
#pragma unroll
      for (int i = 0; i < kTokens * 8; ++i) {
        const float v = wave_reduce_sum(acc[i]);
        if (lane == 0) part[wave][i / 8][i % 8] = v;
      }
    }
    __syncthreads();
    if (threadIdx.x < kTokens * 8) {
      const int t = threadIdx.x / 8, e = threadIdx.x % 8;
      if (e0 + e < E)
        logits[t][e0 + e] = (part[0][t][e] + part[1][t][e]) + (part[2][t][e] + part[3][t][e]);
    }
    __syncthreads();
  }

  const int t = threadIdx.x;
  if (t >= kTokens || t0 + t >= T) return;
  // ties and NaN: the lowest expert that is left, so that every id is an expert
  unsigned long long taken = 0;
  int chosen[kMaxTop];
  float value[kMaxTop], sum = 0.f;
  bool undefined = false;   // a NaN anywhere makes every weight one, as in a full softmax
#pragma unroll
  for (int j = 0; j < kMaxTop; ++j) {
    if (j >= top) break;
    int best = -1;
    float v = 0.f;
    for (int e = 0; e < E; ++e) {
      if (taken >> e & 1) continue;
      const float l = logits[t][e];
      if (j == 0) undefined |= l != l;
      if (best < 0 || l > v) {
        best = e;
        v = l;
      }
    }
    taken |= 1ull << best;
    chosen[j] = best;
    value[j] = v;
  }
  const float most = undefined ? __builtin_nanf("") : value[0];
#pragma unroll
  for (int j = 0; j < kMaxTop; ++j) {
    if (j >= top) break;
    value[j] = __expf(value[j] - most);
    sum += value[j];
  }
#pragma unroll
  for (int j = 0; j < kMaxTop; ++j) {
    if (j >= top) break;
    ids[(long)(t0 + t) * top + j] = chosen[j];
    weights[(long)(t0 + t) * top + j] = value[j] / sum;
  }
}

// Pairs p = t * top + j grouped by expert: seg [E + 1], pos[p] the sorted row of a pair,
// rows[pos[p]] = t; pairs of no expert, whose id is any other, get no row and no pos.  One workgroup:
// a few thousand pairs are less than a second launch.
// Counts and places are claimed in LDS, a pair a lane, but for the lanes of the first one's expert, which
// claims for all of them: where most pairs are of one expert each would wait for the others.  us, a
// wave that claims for the lanes of one expert after the other, a round trip each | each lane for itself |
// here: 33 tokens, 2 of 8 experts 3.7 | 2.2 | 2.2, 2949 15.1 | 4.9 | 5.2, 1000, 8 of 64 87 | 6.7 | 7.5; all of
// one expert, 512 2.4 | 2.8 | 2.3, 4000 4.1 | 8.6 | 3.9; of two 4000 8.4 | 8.6 | 8.8.
__global__ __launch_bounds__(1024) void moe_group_kernel(
    int* __restrict__ rows, int* __restrict__ pos, int* __restrict__ seg,
    const int* __restrict__ ids, const int pairs, const int E, const int top) {
  __shared__ int count[kMaxExperts], next[kMaxExperts];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  for (int e = tid; e < E; e += 1024) count[e] = 0;
  __syncthreads();
  // the lane's place among those of its expert
  auto claim = [&](int* at, int e) {
    const unsigned long long some = __ballot((unsigned)e < (unsigned)E);
    if (some == 0) return 0;
    const int lead = __builtin_ctzll(some), common = __builtin_amdgcn_readlane(e, lead);
    const unsigned long long same = __ballot(e == common);
    int place = 0;
    if (lane == lead || ((unsigned)e < (unsigned)E && e != common))
      place = atomicAdd(&at[e], lane == lead ? __popcll(same) : 1);
    const int ahead = __popcll(same & ((1ull << lane) - 1));
    return e == common ? __builtin_amdgcn_readlane(place, lead) + ahead : place;
  };
  for (int p = tid; p < pairs; p += 1024) claim(count, ids[p]);
  __syncthreads();
  if (tid == 0) {
    int at = 0;
    for (int e = 0; e < E; ++e) {
      seg[e] = at;
      next[e] = at;
      at += count[e];
    }
    seg[E] = at;
  }
  __syncthreads();
  for (int p = tid; p < pairs; p += 1024) {
    const int e = ids[p], row = claim(next, e);
    if ((unsigned)e >= (unsigned)E) continue;
    pos[p] = row;
    rows[row] = p / top;
  }
}

// out[t] = sum_j weights[t, j] ye[pos[t, j]], in f32, rounded once.  Bound by the bytes of ye and
// out, few tokens by the chain from places to rows: eight results a thread, the rows of AHEAD pairs
// asked for at once.  us, 256 threads and a pair after the other | here: 33 x 4096 of 2 2.3 | 1.9, 256
// 3.6 | 2.9, 2949 14.4 | 14.4, 33 x 8192 3.5 | 2.3.  (Four of 8 pairs at once: 33 x 2048 3.0 | 3.2.)
template <int AHEAD>
__global__ __launch_bounds__(1024) void moe_sum_kernel(
    __hip_bfloat16* __restrict__ out,       // [T, H]
    const __hip_bfloat16* __restrict__ ye,  // [T * top, H]
    const int* __restrict__ pos, const float* __restrict__ weights, const int H,
    const int top) {
  const long t = blockIdx.x;
  for (int h = threadIdx.x * 8; h < H; h += blockDim.x * 8) {
    float acc[8] = {};
    for (int j0 = 0; j0 < top; j0 += AHEAD) {
      Vec16<__hip_bfloat16> v[AHEAD];
#pragma unroll
      for (int j = 0; j < AHEAD; ++j)
        v[j] = load16(ye + (long)pos[t * top + min(j0 + j, top - 1)] * H + h);
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        if (j0 + j >= top) break;
        const float w = weights[t * top + j0 + j];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          acc[i] = __builtin_fmaf(w, __bfloat162float(v[j].data[i]), acc[i]);
      }
    }
    Vec16<__hip_bfloat16> o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o.data[i] = __float2bfloat16(acc[i]);
    store16(out + t * H + h, o);
  }
}

}  // namespace

int moe_topk_max_experts() { return kMaxExperts; }
int moe_topk_max_top() { return kMaxTop; }

void launch_moe_topk(int* ids, float* weights, const __hip_bfloat16* x,
                     const __hip_bfloat16* gate, int T, int E, int K, int top,
                     hipStream_t stream) {
  auto go = [&](auto kernel, int tokens) {
    hipLaunchKernelGGL(kernel, dim3((T + tokens - 1) / tokens), dim3(256), 0, stream, ids, weights,
                       x, gate, T, E, K, top);
  };
  // A token a workgroup is the shorter chain, four read the gate matrix once.  us, four | one, 8 experts
  // of 4096 inputs: 1 token 11.1 | 4.9, 33 11.3 | 5.2, 1024 11.9 | 7.7, 2048 12.8 | 11.1, 2949 14.2 | 14.4; 64
  // of 2048: 33 95 | 46, 2000 104 | 78.  (Two: 33 tokens 7.6, 2949 14.2.)  The line is where 8 experts
  // cross; more of them have more sums of a wave to make, which four tokens make one after the other.
  if (T <= 2048) go(moe_topk_kernel<1>, 1);
  else go(moe_topk_kernel<4>, 4);
}

void launch_moe_group(int* rows, int* pos, int* seg, const int* ids, int pairs, int E, int top,
                      hipStream_t stream) {
  hipLaunchKernelGGL(moe_group_kernel, dim3(1), dim3(1024), 0, stream, rows, pos, seg, ids,
                     pairs, E, top);
}

void launch_moe_sum(__hip_bfloat16* out, const __hip_bfloat16* ye, const int* pos,
                    const float* weights, int T, int H, int top, hipStream_t stream) {
  const int threads = H >= 8192 ? 1024 : (H / 8 + 63) / 64 * 64;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(T), dim3(threads), 0, stream, out, ye, pos, weights, H, top);
  };
  if (top <= 2) go(moe_sum_kernel<2>);
  else go(moe_sum_kernel<1>);
}
