// Learned PPE warm start on gfx950 MFMA.
//
// Network: edge MLP e_ij -> 64 -> 64 (ReLU), sum over the neighbour list
// scaled by 1/64, node MLP 64 -> 64 (ReLU) -> 1.
//
// The forward kernel (k_mlp_forward) gives each wave 16 consecutive
// particles and walks their neighbour lists slot by slot, with every layer
// computed transposed so that the 16 MFMA columns are the 16 particles; the
// per-particle sums then stay in registers (layout at the kernel).
//
// The backward kernel owns one particle per wave64, four waves per block, and
// walks its neighbour list in tiles of 16 edges:
//   layer 1  D[16 x 64] = E[16 x 16] W1^T[16 x 64]   4 x v_mfma_f32_16x16x16_bf16
//            (the 6 edge inputs padded to K = 16 with zeros)
//   layer 2  D[16 x 64] = H1[16 x 64] W2^T[64 x 64]  8 x v_mfma_f32_16x16x32_bf16
// MFMA operand layout (16x16x32): lane l holds row (l mod 16) of A and
// column (l mod 16) of B, K elements 8*(l/16) .. 8*(l/16)+7; the FP32
// result holds rows 4*(l/16) .. +3 of column (l mod 16).  The layer-1
// result is re-laid out into the layer-2 A operand through a 16 x 64 BF16
// LDS tile.  The node MLP (64 x 64 per particle, 1/80 of the edge work)
// runs on the VALU with the same BF16 weights.
//
// It is bound by the latency of each wave's chain of gathers, LDS tiles and
// products, with as many waves as the FP32 accumulators leave room for:
//   - a particle's edges are gathered 64 at a time, one per lane, into an LDS
//     list that both passes read (by tiles of 16 lanes, in each pass: 1.58 ms
//     for 64,000 rows; so, with W3 in padded LDS rows: 1.07 ms);
//   - dW3 is shared by the four waves of a block, 16 rows each, and the W2
//     operands lie in LDS, which brings the registers from over 400 to 256, two
//     waves per SIMD (0.85 ms);
//   - the XCDs take runs of particles by turns (0.79 ms).
// Per-particle counts instead of sums for db2 and selects of a rounded dZ2 took
// instructions out but no time.  Half as many blocks, with dW3 written out halfway
// through in place of shorter sums, spilled: 0.87 ms.
//
// Backward recomputes the forward per particle (two passes over its edges)
// and accumulates weight gradients with v_mfma_f32_16x16x16_bf16, whose A
// and B operands are exactly the FP32 result layout above (K = the 16 edges
// of a tile), so dW2 += dZ2^T H1 and dW1 += dZ1^T E need no re-layout.
// dH1 = dZ2 W2 goes through a second LDS tile.  Each block adds its waves'
// FP32 accumulators in FP64 and writes that partial gradient; a second kernel sums
// the partials in a fixed order (deterministic), then Adam updates the FP32 master copy and the
// BF16 copy is refreshed.
#include "learned.hpp"

namespace sophia {

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

// Particles of the backward kernel: one per wave, kBwdWaves per block, the
// blocks of one XCD (workgroups are dealt to XCDs round robin) on consecutive
// ones, so that they share neighbour fields in that XCD's L2.  The XCDs take such
// runs by turns: with one eighth of the particles to each, those with more wall
// particles, which have no row, stood idle for a quarter of the time.
// gridDim.x is a multiple of 8; the trip count is the block's, not the wave's.
constexpr int kBwdWaves = 4;
struct PartIter {
  int i0, stride;
};
__device__ inline PartIter xcd_particles() {
  const int x = blockIdx.x & 7, b = blockIdx.x >> 3, per = gridDim.x >> 3;
  return PartIter{(x * per + b) * kBwdWaves, (int)gridDim.x * kBwdWaves};
}

__device__ inline f4 mfma32(bf8 a, bf8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ inline f4 mfma16(bf4 a, bf4 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0); }

struct Net {
  const __bf16* wbf;
  const float* master;  // biases are read in FP32
};

// Operands of the backward kernel's W2 products, a lane's 16 bytes each, in LDS
// and shared by the block's waves: fragments 2 nb, 2 nb + 1 of layer 2 (B[k][n] =
// W2[n][k], n = nl + 16 nb) and 8 + 2 kb, 8 + 2 kb + 1 of dH1 = dZ2 W2 (B[k = n]
// [col] = W2[n][col], col = nl + 16 kb)
typedef bf8 W2Frags[16][64];

__device__ inline void load_w2_frags(const Net& net, int frag, int lane, W2Frags& F) {
  const int nl = lane & 15, c = nl + 16 * ((frag & 7) >> 1), k0 = 8 * (lane >> 4) + 32 * (frag & 1);
  bf8 t;
#pragma unroll
  for (int j = 0; j < 8; j++) t[j] = net.wbf[OFF_W2 + (frag < 8 ? c * kH + k0 + j : (k0 + j) * kH + c)];
  F[frag][lane] = t;
}

// Edge inputs of up to kEdgeBuf edges of one particle in LDS: row e holds the
// six BF16 inputs of edge e and two zeros (one 16-byte read is a lane's part of
// the layer-1 A operand).
constexpr int kEdgeBuf = 128;
struct EdgeList {
  bf8 e[kEdgeBuf];
};

// Gathers edges base .. base + kEdgeBuf - 1 of particle i, one edge per lane and
// round; returns in valid[q] the edges 64 q + lane that exist.  Inputs of edge
// (i, j): (x_i - x_j)/h_i, |x_i - x_j|/h_i, rho_j/rho_f, s_j.
template <typename R>
__device__ inline void gather_edges(const SphView<R>& v, const float2* nf, int i, int base, int cnt, int lane,
                                    EdgeList& E, uint64_t (&valid)[2]) {
  const double ih = 1.0 / v.h[i];
  const double xi = v.x[i], yi = v.y[i], zi = v.z[i];
#pragma unroll
  for (int q = 0; q < 2; q++) {
    valid[q] = 0;
    if (base + 64 * q >= cnt) continue;
    const int e = base + 64 * q + lane;
    bool ok = false;
    bf8 t;
    for (int k = 0; k < 8; k++) t[k] = (__bf16)0.0f;
    if (e < cnt) {
      const uint32_t ent = v.nbr[nbr_slot(e, i, v.n)];
      if (!(ent & kNbrFlag)) {
        const int j = (int)ent;
        double ex, ey, ez;
        pdiff(v, xi, yi, zi, j, ex, ey, ez);
        const double dx = ex * ih, dy = ey * ih, dz = ez * ih;
        const float2 f = nf[j];
        t[0] = (__bf16)(float)dx;
        t[1] = (__bf16)(float)dy;
        t[2] = (__bf16)(float)dz;
        t[3] = (__bf16)(float)sqrt(dx * dx + dy * dy + dz * dz);
        t[4] = (__bf16)f.x;
        t[5] = (__bf16)f.y;
        ok = true;
      }
    }
    E.e[64 * q + lane] = t;
    valid[q] = __ballot(ok);
  }
}

// layer-1 A operand of tile c of the gathered edges (16x16x16 layout: row l mod
// 16, inputs 4 (l / 16) .. +3, of which 8 .. 15 are zero) and its edge mask
__device__ inline bf4 edge_operand(const EdgeList& E, int c, int lane) {
  bf4 a;
  for (int k = 0; k < 4; k++) a[k] = (__bf16)0.0f;
  if (lane < 32) a = reinterpret_cast<const bf4*>(&E.e[16 * c + (lane & 15)])[lane >> 4];
  return a;
}
__device__ inline uint32_t edge_mask(const uint64_t (&valid)[2], int c) {
  return (uint32_t)((c < 4 ? valid[0] : valid[1]) >> (16 * (c & 3))) & 0xffffu;
}

// layer 1 + ReLU for one tile; z1 in result layout, H (LDS) gets BF16 h1
__device__ inline void layer1(const float (&b1)[4], const bf4 (&B1)[4], bf4 a1, int lane, bf4 (&h1)[4],
                              __bf16 (*H)[kH + 8]) {
  const int nl = lane & 15, er = 4 * (lane >> 4);
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
    f4 z = {0.f, 0.f, 0.f, 0.f};
    z = mfma16(a1, B1[nb], z);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      float hv = fmaxf(z[r] + b1[nb], 0.f);
      __bf16 hb = (__bf16)hv;
      h1[nb][r] = hb;
      H[er + r][nl + 16 * nb] = hb;
    }
  }
}

// layer 2 pre-activation for one tile (A operand read back from H)
__device__ inline void layer2(const W2Frags& F, int lane, __bf16 (*H)[kH + 8], f4 (&z2)[4]) {
  const int e = lane & 15, kq = 8 * (lane >> 4);
  const bf8 a0 = *reinterpret_cast<const bf8*>(&H[e][kq]), a1 = *reinterpret_cast<const bf8*>(&H[e][32 + kq]);
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
    f4 z = {0.f, 0.f, 0.f, 0.f};
    z = mfma32(a0, F[2 * nb][lane], z);
    z = mfma32(a1, F[2 * nb + 1][lane], z);
    z2[nb] = z;
  }
}

// Lanes of one wave exchange the edge inputs through LDS.  A wave's LDS
// instructions execute in issue order, so ordering the compiler's code
// motion with wavefront-scope fences is all the synchronisation needed.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Rows of W3 and of its transpose in LDS: 144 bytes, so the 16-byte reads of
// the 16 lanes of a quarter wave fall on different banks
constexpr int kW3Row = kH + 8;

// node MLP forward: z3 = W3 m + b3 (lane l = output l), y = W4 relu(z3) + b4
__device__ inline float node_forward(const float* Ms, const __bf16 (*W3s)[kW3Row], int lane, float b3, float w4,
                                     float b4, float& z3) {
  float z = b3;
#pragma unroll 2
  for (int k8 = 0; k8 < kH; k8 += 8) {
    const bf8 w = *reinterpret_cast<const bf8*>(&W3s[lane][k8]);
#pragma unroll
    for (int k = 0; k < 8; k++) z += (float)w[k] * Ms[k8 + k];
  }
  z3 = z;
  float y = w4 * fmaxf(z, 0.f);
  for (int off = 32; off > 0; off >>= 1) y += __shfl_xor(y, off);
  return y + b4;
}

// Forward kernel, weights as the A operand.  Each layer is computed
// transposed, Z^T[hidden x 16 edges] = W[hidden x K] E^T[K x 16 edges], so a
// layer's MFMA result (lane l: hidden units 16 nb + 4 (l / 16) + r of edge
// l mod 16) is already the next layer's B operand once the hidden dimension
// is enumerated in that order: K-step s of layer 2 takes, in lane l,
// hidden-1 units 16 (2 s + j / 4) + 4 (l / 16) + j mod 4 (j = 0..7), and the
// W2 A operand is loaded in the same order.  No LDS transpose between the
// layers.  Edge inputs are gathered 64 at a time (one edge per lane) into an
// LDS tile; the messages are summed per lane over the tiles and then over
// the 16 lanes of each group.  Biases are added in FP32 after each MFMA, as
// in the backward kernel's recomputation.
struct FwdOperands {
  bf4 A1[4];      // W1 rows 16 nb + (l mod 16), inputs 4 (l / 16) .. +3 (16x16x16 layout): K = 0..5 the
                  // edge inputs, K = 6, 7 the BF16 high and low parts of b1 (inputs 6, 7 are 1), rest 0
  bf8 A2[4][2];   // W2 rows 16 mb + (l mod 16), hidden-1 units in the layer-1 result order
  f4 C2[4];       // b2 in the layer-2 result layout (units 16 mb + 4 (l / 16) + r), the accumulator start
};

__device__ inline void load_fwd_t(const Net& net, int lane, FwdOperands& w) {
  const int m = lane & 15, g = lane >> 4;
#pragma unroll
  for (int nb = 0; nb < 4; nb++) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int k = 4 * g + j;
      const float b1 = net.master[OFF_B1 + 16 * nb + m];
      const __bf16 b1h = (__bf16)b1;
      w.A1[nb][j] = k < kEin ? net.wbf[OFF_W1 + (16 * nb + m) * kEin + k]
                  : k == kEin ? b1h : k == kEin + 1 ? (__bf16)(b1 - (float)b1h) : (__bf16)0.0f;
    }
  }
#pragma unroll
  for (int mb = 0; mb < 4; mb++)
#pragma unroll
    for (int sk = 0; sk < 2; sk++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const int u = 16 * (2 * sk + j / 4) + 4 * g + (j & 3);
        w.A2[mb][sk][j] = net.wbf[OFF_W2 + (16 * mb + m) * kH + u];
      }
#pragma unroll
  for (int mb = 0; mb < 4; mb++)
#pragma unroll
    for (int r = 0; r < 4; r++) w.C2[mb][r] = net.master[OFF_B2 + 16 * mb + 4 * g + r];
}

// ReLU through the sign bit: an integer max with 0 maps every negative
// float (and -0) to +0 and leaves the rest unchanged, without the NaN
// canonicalisation a float max needs
__device__ inline float relu_bits(float x) { return __int_as_float(max(__float_as_int(x), 0)); }
// ReLU of two BF16 values packed in one dword (integer max per half)
__device__ inline uint32_t relu_pk_bf16(float a, float b) {
  typedef short s2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
  typedef float fl2 __attribute__((ext_vector_type(2)));
  const fl2 f = {a, b};
  const s2 v = __builtin_bit_cast(s2, __builtin_convertvector(f, bf2));
  const s2 z = {0, 0};
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(v, z));
}

constexpr int kFwdWaves = 4;    // waves per block of the forward kernel

// Group of 16 particles of this wave.  Blocks are dealt to XCDs round robin; an
// XCD takes runs of kFwdRun blocks (1024 consecutive particles), so that the groups
// it works on at one time share neighbour fields in its L2, and the XCDs take such
// runs by turns, since wall particles lie together and cost nothing.  One group per
// wave, so that a free slot takes the next block: at 1.16 M particles 998 us, 1066
// with 1024 persistent blocks, 1088 with one eighth of the particles to each XCD.
constexpr int kFwdRun = 16;
__device__ inline int fwd_group() {
  const int k = (int)blockIdx.x >> 3, x = (int)blockIdx.x & 7;
  return (((k / kFwdRun) * 8 + x) * kFwdRun + k % kFwdRun) * kFwdWaves + (int)(threadIdx.x >> 6);
}

// Forward kernel.  One wave owns a group of 16 consecutive particles and
// walks their neighbour lists slot by slot, four slots per gather round
// (lane l gathers the edge of particle l mod 16 at slot k0 + l / 16).  Each
// layer is computed transposed, Z^T[hidden x 16] = W[hidden x K] E^T[K x 16],
// with the 16 MFMA columns being the group's 16 particles at one slot:
//   - a layer's result (lane l: hidden units 16 nb + 4 (l / 16) + r of
//     particle l mod 16) is the next layer's B operand once the hidden
//     dimension is enumerated in that order (K-step s of the next layer
//     takes, in lane l, units 16 (2 s + j / 4) + 4 (l / 16) + j mod 4,
//     j = 0..7; the A operand holds the weights in the same order);
//   - the ReLU messages are summed over the slots in registers, so the
//     aggregated message of particle l mod 16 ends up spread over the four
//     lanes l mod 16 + 16 q with no cross-lane reduction, already in the
//     node layer's B-operand order.
// The node layer runs on MFMA as well: the FP32 message is split into BF16
// high and low parts (hi + lo equals it to 2^-16 relative), so the result
// matches an FP32 message against the BF16 weights W3.  Each edge carries
// two extra inputs equal to 1 (0 for a slot past the particle's list), and
// b1 enters layer 1 as its BF16 high and low parts against them; a slot with
// no edge then has h1 = 0 exactly.  Layer 2 starts its accumulation from b2
// (FP32), so an absent edge adds exactly ReLU(b2), which is taken off once
// per particle at the end: no per-slot masking.  b3 is added in FP32.  Edge
// inputs use the pos4 position records.
template <typename R>
__global__ __launch_bounds__(64 * kFwdWaves, 4) void k_mlp_forward(Net net, SphView<R> v,
                                                                   const float2* __restrict__ nf,
                                                                   const int* __restrict__ row,
                                                                   const double* __restrict__ pprev, double scale,
                                                                   double* __restrict__ guess) {
  __shared__ bf8 A3s[4][2][64];                         // W3 as the node layer's A operand, per lane
  __shared__ __attribute__((aligned(16))) float bs[2 * kH];  // b3, W4 (W4 from its BF16 copy)
  __shared__ bf8 Et[kFwdWaves][64];                     // edge inputs of one gather round, per wave
  const int tid = threadIdx.x, lane = tid & 63;
  const int m = lane & 15, g4 = lane >> 4;
  for (int q = tid; q < 4 * 2 * 64; q += blockDim.x) {
    const int mb = q >> 7, sk = (q >> 6) & 1, l = q & 63;
    bf8 a;
#pragma unroll
    for (int j = 0; j < 8; j++)
      a[j] = net.wbf[OFF_W3 + (16 * mb + (l & 15)) * kH + 16 * (2 * sk + j / 4) + 4 * (l >> 4) + (j & 3)];
    A3s[mb][sk][l] = a;
  }
  if (tid < kH) {
    bs[tid] = net.master[OFF_B3 + tid];
    bs[kH + tid] = (float)net.wbf[OFF_W4 + tid];
  }
  FwdOperands w;
  load_fwd_t(net, lane, w);
  __syncthreads();
  bf8* E = Et[tid >> 6];
  const bf4* E4 = reinterpret_cast<const bf4*>(E);  // inputs 0-3 and 4-7 of each edge
  const float b4 = net.master[OFF_B4];
  const int i = fwd_group() * 16 + m;
  const bool live = i < v.n;
  const bool isrow = live && row[i] != 0;
  const int cnt = isrow ? min(v.nbr_cnt[i], v.nbr_cap) : 0;
  int maxc = cnt;
#pragma unroll
  for (int off = 1; off < 16; off <<= 1) maxc = max(maxc, __shfl_xor(maxc, off));
  float y = 0.f;
  if (__ballot(isrow) != 0) {  // wave-uniform
    const float4 pi = isrow ? v.pos4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float ih = isrow ? (float)(1.0 / (double)v.h[i]) : 0.f;
    float acc[4][4] = {};
    int nvalid = 0;  // edges this lane gathered (particle l mod 16)
    uint32_t nxt = g4 < cnt ? v.nbr[nbr_slot(g4, i, v.n)] : kNbrFlag;
    for (int k0 = 0; k0 < maxc; k0 += 4) {
      const uint32_t ent = nxt;
      const int kn = k0 + 4 + g4;
      if (k0 + 4 < maxc) nxt = kn < cnt ? v.nbr[nbr_slot(kn, i, v.n)] : kNbrFlag;
      // an edge outside the list gets all-zero inputs, bias inputs included, so
      // its h1 is exactly 0 and it adds ReLU(b2), taken off after the last slot
      bf8 e8;
#pragma unroll
      for (int q = 0; q < 8; q++) e8[q] = (__bf16)0.0f;
      if (!(ent & kNbrFlag)) {
        nvalid++;
        const int j = (int)ent;
        const float4 pj = v.pos4[j];
        const float2 f = nf[j];
        const float3 d = rel_diff(pi, pj, v.pgrid, v.pmask);
        const float dx = d.x * ih, dy = d.y * ih, dz = d.z * ih;
        e8[0] = (__bf16)dx;
        e8[1] = (__bf16)dy;
        e8[2] = (__bf16)dz;
        e8[3] = (__bf16)__builtin_amdgcn_sqrtf(dx * dx + dy * dy + dz * dz);
        e8[4] = (__bf16)f.x;
        e8[5] = (__bf16)f.y;
        e8[6] = (__bf16)1.0f;  // bias inputs
        e8[7] = (__bf16)1.0f;
      }
      wave_lds_sync();  // the previous round's reads of E are issued
      E[lane] = e8;
      wave_lds_sync();
#pragma unroll 2
      for (int t = 0; t < 4; t++) {
        bf4 b;
#pragma unroll
        for (int q = 0; q < 4; q++) b[q] = (__bf16)0.0f;
        if (g4 < 2) b = E4[2 * (16 * t + m) + g4];
        // layer 1 (16 hidden x 16 particles per block nb, K = 16, b1
        // included), ReLU, packed straight into the layer-2 B operand
        uint32_t B2u[2][4];
#pragma unroll
        for (int nb = 0; nb < 4; nb++) {
          f4 z = {0.f, 0.f, 0.f, 0.f};
          z = mfma16(w.A1[nb], b, z);
          B2u[nb >> 1][2 * (nb & 1) + 0] = relu_pk_bf16(z[0], z[1]);
          B2u[nb >> 1][2 * (nb & 1) + 1] = relu_pk_bf16(z[2], z[3]);
        }
        const bf8 B20 = __builtin_bit_cast(bf8, B2u[0]), B21 = __builtin_bit_cast(bf8, B2u[1]);
        // layer 2 from b2, ReLU and the sum over slots; an absent edge
        // (h1 = 0) adds ReLU(b2), taken off after the last slot
#pragma unroll
        for (int mb = 0; mb < 4; mb++) {
          f4 z = mfma32(w.A2[mb][0], B20, w.C2[mb]);
          z = mfma32(w.A2[mb][1], B21, z);
          acc[mb][0] += relu_bits(z[0]);
          acc[mb][1] += relu_bits(z[1]);
          acc[mb][2] += relu_bits(z[2]);
          acc[mb][3] += relu_bits(z[3]);
        }
      }
    }
    {
      // absent edges among the 4 * rounds slots processed per particle
      int nv = nvalid;
      nv += __shfl_xor(nv, 16);
      nv += __shfl_xor(nv, 32);
      const float absent = (float)(((maxc + 3) & ~3) - nv);
#pragma unroll
      for (int mb = 0; mb < 4; mb++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[mb][r] -= absent * relu_bits(w.C2[mb][r]);
    }
    // node layer: message M = acc / 64 as BF16 hi + lo parts
    bf8 Bh[2], Bl[2];
#pragma unroll
    for (int sk = 0; sk < 2; sk++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float mv = acc[2 * sk + j / 4][j & 3] * (1.0f / 64.0f);
        const __bf16 hb = (__bf16)mv;
        Bh[sk][j] = hb;
        Bl[sk][j] = (__bf16)(mv - (float)hb);
      }
    float yp = 0.f;
#pragma unroll
    for (int mb = 0; mb < 4; mb++) {
      const bf8 a0 = A3s[mb][0][lane], a1 = A3s[mb][1][lane];
      f4 z = {0.f, 0.f, 0.f, 0.f};
      z = mfma32(a0, Bl[0], z);
      z = mfma32(a1, Bl[1], z);
      z = mfma32(a0, Bh[0], z);
      z = mfma32(a1, Bh[1], z);
      const float4 bb = *reinterpret_cast<const float4*>(bs + 16 * mb + 4 * g4);
      const float4 ww = *reinterpret_cast<const float4*>(bs + kH + 16 * mb + 4 * g4);
      yp += ww.x * fmaxf(z[0] + bb.x, 0.f) + ww.y * fmaxf(z[1] + bb.y, 0.f) + ww.z * fmaxf(z[2] + bb.z, 0.f) +
            ww.w * fmaxf(z[3] + bb.w, 0.f);
    }
    yp += __shfl_xor(yp, 16);
    yp += __shfl_xor(yp, 32);
    y = yp + b4;
  }
  if (g4 == 0 && live) guess[i] = isrow ? pprev[i] + scale * (double)y : pprev[i];
}

template <typename R>
__global__ __launch_bounds__(64 * kBwdWaves, 2) void k_mlp_backward(Net net, SphView<R> v, const float2* __restrict__ nf,
                                                      const int* __restrict__ row, const double* __restrict__ pprev,
                                                      const double* __restrict__ target, double inv_scale,
                                                      float inv_rows, double* __restrict__ partials) {
  struct Work {
    W2Frags F;
    EdgeList E[kBwdWaves];
    alignas(16) __bf16 H[kBwdWaves][16][kH + 8];
    alignas(16) __bf16 DZ[kBwdWaves][16][kH + 8];
    alignas(16) __bf16 W3s[kH][kW3Row];  // W3[l][k]
    alignas(16) __bf16 W3t[kH][kW3Row];  // W3[l][k] at [k][l]
    alignas(16) float DM[kBwdWaves][kH];
    alignas(16) float Ms[2][kBwdWaves][kH];  // by turns, so that one barrier an iteration is enough
    alignas(16) float DG[2][kBwdWaves][kH];
  };
  __shared__ union {
    Work w;
    double grad[kNParam + 1];  // the block's partial gradient, after the loop
  } sh;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nl = lane & 15, er = 4 * (lane >> 4), kq = 8 * (lane >> 4);
  auto& W3s = sh.w.W3s;
  auto& W3t = sh.w.W3t;
  W2Frags& F = sh.w.F;
  EdgeList& E = sh.w.E[wave];
  auto& H = sh.w.H[wave];
  auto& DZ = sh.w.DZ[wave];
  auto& DM = sh.w.DM[wave];
  for (int q = threadIdx.x; q < kH * kH; q += 64 * kBwdWaves) {
    const __bf16 w = net.wbf[OFF_W3 + q];
    W3s[q / kH][q % kH] = w;
    W3t[q % kH][q / kH] = w;
  }
  for (int f = wave; f < 16; f += kBwdWaves) load_w2_frags(net, f, lane, F);
  bf4 B1[4];  // B[k][n] = W1[n][k], k < 6
  float b1[4], b2[4];
#pragma unroll
  for (int kb = 0; kb < 4; kb++) {
#pragma unroll
    for (int j = 0; j < 4; j++)
      B1[kb][j] = er + j < kEin ? net.wbf[OFF_W1 + (nl + 16 * kb) * kEin + er + j] : (__bf16)0.0f;
    b1[kb] = net.master[OFF_B1 + nl + 16 * kb];
    b2[kb] = net.master[OFF_B2 + nl + 16 * kb];
  }
  const float w4 = (float)net.wbf[OFF_W4 + lane], b3 = net.master[OFF_B3 + lane], b4 = net.master[OFF_B4];
  __syncthreads();

  f4 gW2[16], gW1[4];
#pragma unroll
  for (int q = 0; q < 16; q++) gW2[q] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 4; q++) gW1[q] = (f4){0.f, 0.f, 0.f, 0.f};
  float gb1[4] = {0, 0, 0, 0}, gb2[4] = {0, 0, 0, 0};
  // rows 16 wave .. + 15 of dW3, column = lane
  float gW3[16];
#pragma unroll
  for (int k = 0; k < 16; k++) gW3[k] = 0.f;
  float gb3 = 0.f, gW4 = 0.f, gb4 = 0.f, loss = 0.f;

  int turn = 0;
  for (PartIter it = xcd_particles(); it.i0 < v.n; it.i0 += it.stride, turn ^= 1) {
    const int i = it.i0 + wave;
    const bool live = i < v.n && row[i];
    float* Ms = sh.w.Ms[turn][wave];
    float* DG = sh.w.DG[turn][wave];
    const int cnt = live ? min(v.nbr_cnt[i], v.nbr_cap) : 0;
    uint64_t valid[2] = {0, 0};
    // pass 1: forward, the message summed over the edges
    if (live) {
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
      for (int base = 0; base < cnt; base += kEdgeBuf) {
        gather_edges(v, nf, i, base, cnt, lane, E, valid);
        wave_lds_sync();
        for (int c = 0; c < kEdgeBuf / 16 && base + c * 16 < cnt; c++) {
          const uint32_t on = edge_mask(valid, c);
          bf4 h1[4];
          f4 z2[4];
          layer1(b1, B1, edge_operand(E, c, lane), lane, h1, H);
          wave_lds_sync();
          layer2(F, lane, H, z2);
#pragma unroll
          for (int nb = 0; nb < 4; nb++)
#pragma unroll
            for (int r = 0; r < 4; r++)
              if ((on >> (er + r)) & 1u) acc[nb] += fmaxf(z2[nb][r] + b2[nb], 0.f);
          wave_lds_sync();
        }
      }
#pragma unroll
      for (int nb = 0; nb < 4; nb++) {
        acc[nb] += __shfl_xor(acc[nb], 16);
        acc[nb] += __shfl_xor(acc[nb], 32);
      }
      if (lane < 16) {
#pragma unroll
        for (int nb = 0; nb < 4; nb++) Ms[lane + 16 * nb] = acc[nb] * (1.0f / 64.0f);
      }
      wave_lds_sync();
    float z3;
    const float y = node_forward(Ms, W3s, lane, b3, w4, b4, z3);
    const float t = (float)((target[i] - pprev[i]) * inv_scale);
    const float err = y - t;
    const float dy = 2.f * err * inv_rows;
    if (lane == 0) {
      loss += err * err * inv_rows;
      gb4 += dy;
    }
    const float g = fmaxf(z3, 0.f);
    gW4 += dy * g;
    const float dg = z3 > 0.f ? dy * w4 : 0.f;
    gb3 += dg;
    DG[lane] = dg;
    } else {
      Ms[lane] = 0.f;
      DG[lane] = 0.f;
    }
    // dW3 += dG M^T of the block's particles, each wave its 16 rows
    __syncthreads();
#pragma unroll
    for (int p = 0; p < kBwdWaves; p++) {
      const float mk = sh.w.Ms[turn][p][lane];
#pragma unroll
      for (int r4 = 0; r4 < 16; r4 += 4) {
        const float4 d = *reinterpret_cast<const float4*>(&sh.w.DG[turn][p][16 * wave + r4]);
        gW3[r4 + 0] += d.x * mk;
        gW3[r4 + 1] += d.y * mk;
        gW3[r4 + 2] += d.z * mk;
        gW3[r4 + 3] += d.w * mk;
      }
    }
    if (!live) continue;
    {
      float dm = 0.f;
#pragma unroll 2
      for (int l8 = 0; l8 < kH; l8 += 8) {
        const bf8 w = *reinterpret_cast<const bf8*>(&W3t[lane][l8]);
#pragma unroll
        for (int l = 0; l < 8; l++) dm += (float)w[l] * DG[l8 + l];
      }
      DM[lane] = dm * (1.0f / 64.0f);
    }
    wave_lds_sync();
    float dmv[4];
#pragma unroll
    for (int nb = 0; nb < 4; nb++) dmv[nb] = DM[nl + 16 * nb];
    // pass 2: edge backward; a list of up to kEdgeBuf edges is still in E
    for (int base = 0; base < cnt; base += kEdgeBuf) {
      if (cnt > kEdgeBuf) {
        gather_edges(v, nf, i, base, cnt, lane, E, valid);
        wave_lds_sync();
      }
      for (int c = 0; c < kEdgeBuf / 16 && base + c * 16 < cnt; c++) {
        const uint32_t valid16 = edge_mask(valid, c);
        bf4 h1[4];
        layer1(b1, B1, edge_operand(E, c, lane), lane, h1, H);
        wave_lds_sync();
        f4 z2[4];
        layer2(F, lane, H, z2);
        // dZ2 in result layout; edges outside the list contribute nothing
        f4 dz2[4];
#pragma unroll
        for (int nb = 0; nb < 4; nb++) {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const bool on = ((valid16 >> (er + r)) & 1u) && (z2[nb][r] + b2[nb] > 0.f);
            const float d = on ? dmv[nb] : 0.f;
            dz2[nb][r] = d;
            gb2[nb] += d;
            DZ[er + r][nl + 16 * nb] = (__bf16)d;
          }
        }
        // dW2 tiles: A = dZ2 (rows n, K = edges), B = H1 (K = edges, cols k)
#pragma unroll
        for (int nb = 0; nb < 4; nb++) {
          bf4 a;
          for (int r = 0; r < 4; r++) a[r] = (__bf16)dz2[nb][r];
#pragma unroll
          for (int kb = 0; kb < 4; kb++) gW2[nb * 4 + kb] = mfma16(a, h1[kb], gW2[nb * 4 + kb]);
        }
        wave_lds_sync();
        // dH1 = dZ2 W2 (A from the DZ tile), then dZ1 through the ReLU
        const bf8 ad0 = *reinterpret_cast<const bf8*>(&DZ[nl][kq]);
        const bf8 ad1 = *reinterpret_cast<const bf8*>(&DZ[nl][32 + kq]);
        bf4 be;
        for (int r = 0; r < 4; r++)
          be[r] = nl < 8 ? reinterpret_cast<const __bf16*>(&E.e[16 * c + er + r])[nl & 7] : (__bf16)0.0f;
#pragma unroll
        for (int kb = 0; kb < 4; kb++) {
          f4 dh = {0.f, 0.f, 0.f, 0.f};
          dh = mfma32(ad0, F[8 + 2 * kb][lane], dh);
          dh = mfma32(ad1, F[8 + 2 * kb + 1][lane], dh);
          bf4 a;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const bool on = ((valid16 >> (er + r)) & 1u) && (float)h1[kb][r] > 0.f;
            const float d = on ? dh[r] : 0.f;
            gb1[kb] += d;
            a[r] = (__bf16)d;
          }
          gW1[kb] = mfma16(a, be, gW1[kb]);
        }
        wave_lds_sync();
      }
    }
  }
  // the block's partial gradient: the waves add theirs in turn, in FP64
  __syncthreads();
  for (int q = threadIdx.x; q <= kNParam; q += 64 * kBwdWaves) sh.grad[q] = 0.0;
  for (int w = 0; w < kBwdWaves; w++) {
    __syncthreads();
    if (wave == w) {
      double* P = sh.grad;
      auto put = [&](int q, double a) { P[q] += a; };
#pragma unroll
      for (int nb = 0; nb < 4; nb++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
          const int n = 16 * nb + er + jj;
          if (nl < kEin) put(OFF_W1 + n * kEin + nl, gW1[nb][jj]);
#pragma unroll
          for (int kb = 0; kb < 4; kb++) put(OFF_W2 + n * kH + 16 * kb + nl, gW2[nb * 4 + kb][jj]);
        }
#pragma unroll
      for (int nb = 0; nb < 4; nb++) {
        double a = gb1[nb], b = gb2[nb];
        a += __shfl_xor(a, 16);
        a += __shfl_xor(a, 32);
        b += __shfl_xor(b, 16);
        b += __shfl_xor(b, 32);
        if (lane < 16) {
          put(OFF_B1 + lane + 16 * nb, a);
          put(OFF_B2 + lane + 16 * nb, b);
        }
      }
#pragma unroll
      for (int r = 0; r < 16; r++) P[OFF_W3 + (16 * w + r) * kH + lane] = gW3[r];
      put(OFF_B3 + lane, gb3);
      put(OFF_W4 + lane, gW4);
      if (lane == 0) {
        put(OFF_B4, gb4);
        put(kNParam, loss);
      }
    }
  }
  __syncthreads();
  double* P = partials + (size_t)blockIdx.x * (kNParam + 1);
  for (int q = threadIdx.x; q <= kNParam; q += 64 * kBwdWaves) P[q] = sh.grad[q];
}

// Sum of the blocks' partial gradients in FP64, in a fixed order: 64 parameters
// per block by 16 slices of the partials, so that they are read by 139
// blocks of 16 waves (one thread per parameter walking 1024 partials of 35 KB took
// 260 us, 139 waves with one load in flight each; now 15 us for 1024 of 71 KB).
constexpr int kRedSlices = 16;
__global__ __launch_bounds__(64 * kRedSlices) void k_reduce_partials(const double* __restrict__ partials, int nblocks,
                                                                     float* __restrict__ grad,
                                                                     double* __restrict__ loss) {
  __shared__ double part[kRedSlices][64];
  const int l = threadIdx.x & 63, sl = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + l;
  double s = 0;
  if (p <= kNParam) {
#pragma unroll 8
    for (int b = sl; b < nblocks; b += kRedSlices) s += partials[(size_t)b * (kNParam + 1) + p];
  }
  part[sl][l] = s;
  __syncthreads();
  if (sl != 0 || p > kNParam) return;
  for (int q = 1; q < kRedSlices; q++) s += part[q][l];
  if (p < kNParam) grad[p] = (float)s;
  else *loss = s;
}

// one Adam step; skipped as a whole when the batch loss is not finite, so a
// single bad batch cannot poison the weights
__global__ void k_adam(float* w, const float* g, float* m, float* v, int n, float lr, float b1t, float b2t,
                       const double* loss) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || !isfinite(*loss)) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  float gm = b1 * m[p] + (1.f - b1) * g[p];
  float gv = b2 * v[p] + (1.f - b2) * g[p] * g[p];
  m[p] = gm;
  v[p] = gv;
  float mh = gm / (1.f - b1t), vh = gv / (1.f - b2t);
  w[p] -= lr * mh / (sqrtf(vh) + eps);
}

__global__ void k_to_bf16(const float* w, __bf16* o, int n) {
  int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) o[p] = (__bf16)w[p];
}

// sums over rows of r0^2 and diag, and the row count: per-block partials
// (grid-stride), then one block adds them in a fixed order -> scal[0..2]
constexpr int kFeatBlocks = 256;
__device__ inline double block_sum256(double a, double* sh) {
  for (int off = 32; off > 0; off >>= 1) a += __shfl_xor(a, off);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = a;
  __syncthreads();
  return sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ __launch_bounds__(256) void k_feature_partials(int n, const int* row, const double* r0, const double* diag,
                                                          double* part) {
  __shared__ double sh[4];
  double a = 0, b = 0, c = 0;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    if (row[i]) {
      a += r0[i] * r0[i];
      b += diag[i];
      c += 1;
    }
  a = block_sum256(a, sh);
  b = block_sum256(b, sh);
  c = block_sum256(c, sh);
  if (threadIdx.x == 0) {
    part[3 * blockIdx.x + 0] = a;
    part[3 * blockIdx.x + 1] = b;
    part[3 * blockIdx.x + 2] = c;
  }
}

__global__ __launch_bounds__(256) void k_feature_fin(const double* part, int nb, double* scal) {
  __shared__ double sh[4];
  for (int q = 0; q < 3; q++) {
    double a = 0;
    for (int k = threadIdx.x; k < nb; k += 256) a += part[3 * k + q];
    a = block_sum256(a, sh);
    if (threadIdx.x == 0) scal[q] = a;
  }
}

template <typename R>
__global__ void k_node_features(int n, const int* row, const double* r0, const double* rho, double rho_f,
                                double inv_rms, float2* nf) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  nf[i] = make_float2((float)(rho[i] / rho_f), row[i] ? (float)(r0[i] * inv_rms) : 0.f);
}

__global__ void k_prev(int n, const int* row, const double* pres, double* x) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = row[i] ? pres[i] : 0.0;
}

}  // namespace

int mlp_param_count() { return kNParam; }

int mlp_alloc(Mlp& m, int n, int cap) {
  size_t N = (size_t)(n > 0 ? n : 1);
  if (!m.master) {
    HIP_TRY(hipMalloc(&m.master, kNParam * 4));
    HIP_TRY(hipMalloc(&m.grad, kNParam * 4));
    HIP_TRY(hipMalloc(&m.adam_m, kNParam * 4));
    HIP_TRY(hipMalloc(&m.adam_v, kNParam * 4));
    HIP_TRY(hipMalloc(&m.wbf, kNParam * 2));
    HIP_TRY(hipMalloc(&m.partials, (size_t)kMlpBwdBlocks * (kNParam + 1) * 8));
    HIP_TRY(hipMalloc(&m.scal, 8 * 8));
    HIP_TRY(hipMalloc(&m.fpart, kFeatBlocks * 3 * 8));
    HIP_TRY(hipHostMalloc((void**)&m.host_scal, 8 * 8, hipHostMallocDefault));
  }
  if (m.n != n || !m.nf) {
    if (m.nf) (void)hipFree(m.nf);
    if (m.r0) (void)hipFree(m.r0);
    if (m.guess) (void)hipFree(m.guess);
    if (m.target) (void)hipFree(m.target);
    if (m.pprev) (void)hipFree(m.pprev);
    HIP_TRY(hipMalloc(&m.pprev, N * 8));
    HIP_TRY(hipMalloc(&m.nf, N * sizeof(float2)));
    HIP_TRY(hipMalloc(&m.r0, N * 8));
    HIP_TRY(hipMalloc(&m.guess, N * 8));
    HIP_TRY(hipMalloc(&m.target, N * 8));
  }
  m.n = n;
  m.cap = cap;
  return 0;
}

void mlp_free(Mlp& m) {
  for (void* p : {(void*)m.master, (void*)m.grad, (void*)m.adam_m, (void*)m.adam_v, (void*)m.wbf, (void*)m.partials,
                  (void*)m.scal, (void*)m.fpart, (void*)m.nf, (void*)m.r0, (void*)m.guess, (void*)m.target, (void*)m.pprev})
    if (p) (void)hipFree(p);
  if (m.host_scal) (void)hipHostFree(m.host_scal);
  m = Mlp{};
}

int mlp_set_params(hipStream_t s, Mlp& m, const float* host, int n) {
  if (n != kNParam) {
    set_error("mlp_set_params: %d parameters given, network has %d", n, kNParam);
    return SOPHIA_E_ARG;
  }
  HIP_TRY(hipMemcpyAsync(m.master, host, kNParam * 4, hipMemcpyHostToDevice, s));
  k_to_bf16<<<grid_for(kNParam), kBlock, 0, s>>>(m.master, m.wbf, kNParam);
  HIP_TRY(hipGetLastError());
  int rc = mlp_reset_adam(s, m);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(s));
  m.ready = true;
  return 0;
}

int mlp_get_params(hipStream_t s, const Mlp& m, float* host, int n) {
  if (n != kNParam) {
    set_error("mlp_get_params: buffer of %d, network has %d", n, kNParam);
    return SOPHIA_E_ARG;
  }
  if (!m.ready) {
    set_error("mlp_get_params: parameters not set");
    return SOPHIA_E_STATE;
  }
  HIP_TRY(hipMemcpyAsync(host, m.master, kNParam * 4, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  return 0;
}

int mlp_reset_adam(hipStream_t s, Mlp& m) {
  if (!m.adam_m) return 0;
  int rc = fill_zero_bytes(s, m.adam_m, kNParam * 4);
  if (!rc) rc = fill_zero_bytes(s, m.adam_v, kNParam * 4);
  m.adam_t = 0;
  return rc;
}

template <typename R>
int mlp_features(hipStream_t s, const DevParams& P, const SphView<R>& v, Mlp& m, const int* row, const double* diag,
                 double* scale, double* rr_base) {
  if (v.n <= 0) {
    *scale = 1;
    if (rr_base) *rr_base = 0;
    return 0;
  }
  const int nb = std::min(kFeatBlocks, (v.n + 255) / 256);
  k_feature_partials<<<nb, 256, 0, s>>>(v.n, row, m.r0, diag, m.fpart);
  k_feature_fin<<<1, 256, 0, s>>>(m.fpart, nb, m.scal);
  HIP_TRY(hipMemcpyAsync(m.host_scal, m.scal, 3 * 8, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  if (rr_base) *rr_base = m.host_scal[0];  // sum of r0^2 over the rows
  const double rows = m.host_scal[2] > 0 ? m.host_scal[2] : 1;
  double rms = sqrt(m.host_scal[0] / rows);
  const double dmean = m.host_scal[1] / rows;
  if (!(rms > 0)) rms = 1e-300;
  *scale = dmean > 0 ? rms / dmean : 0.0;
  k_node_features<R><<<grid_for(v.n), kBlock, 0, s>>>(v.n, row, m.r0, v.rho, P.rho_fluid, 1.0 / rms, m.nf);
  HIP_TRY(hipGetLastError());
  return 0;
}

template <typename R>
int mlp_forward(hipStream_t s, const DevParams& P, const SphView<R>& v, Mlp& m, const int* row, const double* pprev,
                double scale, double* guess) {
  if (!m.ready) {
    set_error("learned warm start: parameters not set");
    return SOPHIA_E_STATE;
  }
  if (v.n <= 0) return 0;
  Net net{m.wbf, m.master};
  constexpr int turn = 8 * kFwdRun;  // blocks of one run on each XCD
  const int g = ((v.n + 16 * kFwdWaves - 1) / (16 * kFwdWaves) + turn - 1) / turn * turn;
  k_mlp_forward<R><<<g, 64 * kFwdWaves, 0, s>>>(net, v, m.nf, row, pprev, scale, guess);
  HIP_TRY(hipGetLastError());
  return 0;
}

template <typename R>
int mlp_backward(hipStream_t s, const DevParams& P, const SphView<R>& v, Mlp& m, const int* row, const double* pprev,
                 const double* target, double scale, int n_rows, bool step, double lr, double* loss) {
  if (!m.ready) {
    set_error("learned warm start: parameters not set");
    return SOPHIA_E_STATE;
  }
  if (v.n <= 0 || n_rows <= 0) return 0;
  Net net{m.wbf, m.master};
  // no more blocks than have particles; a multiple of 8, for the XCDs
  const int g = std::min(kMlpBwdBlocks, ((v.n + kBwdWaves - 1) / kBwdWaves + 7) / 8 * 8);
  const double inv_scale = scale != 0 ? 1.0 / scale : 0.0;
  k_mlp_backward<R><<<g, 64 * kBwdWaves, 0, s>>>(net, v, m.nf, row, pprev, target, inv_scale, 1.0f / (float)n_rows,
                                     m.partials);
  k_reduce_partials<<<(kNParam + 1 + 63) / 64, 64 * kRedSlices, 0, s>>>(m.partials, g, m.grad, m.scal + 4);
  HIP_TRY(hipGetLastError());
  if (step) {
    m.adam_t += 1;
    const float b1t = (float)pow(0.9, m.adam_t), b2t = (float)pow(0.999, m.adam_t);
    k_adam<<<grid_for(kNParam), kBlock, 0, s>>>(m.master, m.grad, m.adam_m, m.adam_v, kNParam, (float)lr, b1t, b2t,
                                                 m.scal + 4);
    k_to_bf16<<<grid_for(kNParam), kBlock, 0, s>>>(m.master, m.wbf, kNParam);
    HIP_TRY(hipGetLastError());
  }
  if (loss) {
    HIP_TRY(hipMemcpyAsync(m.host_scal + 4, m.scal + 4, 8, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    *loss = m.host_scal[4];
  }
  return 0;
}

int mlp_gather_previous(hipStream_t s, int n, const int* row, const double* pres, double* x) {
  if (n <= 0) return 0;
  k_prev<<<grid_for(n), kBlock, 0, s>>>(n, row, pres, x);
  HIP_TRY(hipGetLastError());
  return 0;
}

#define INST(R)                                                                                                    \
  template int mlp_features<R>(hipStream_t, const DevParams&, const SphView<R>&, Mlp&, const int*, const double*, \
                               double*, double*);                                                                 \
  template int mlp_forward<R>(hipStream_t, const DevParams&, const SphView<R>&, Mlp&, const int*, const double*,  \
                              double, double*);                                                                   \
  template int mlp_backward<R>(hipStream_t, const DevParams&, const SphView<R>&, Mlp&, const int*, const double*, \
                               const double*, double, int, bool, double, double*);
INST(float)
INST(double)

}  // namespace sophia
