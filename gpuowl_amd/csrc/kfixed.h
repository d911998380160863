// Shape-specialized row and column passes for gfx950 (templates; the kfix_*.hip files
// instantiate them for the compiled shapes and export their name tables).
//
// Same algorithm, layout and modes as k_row / k_col in kernels.hip, with the
// FFT plan fixed at compile time (no integer division, no radix dispatch, every
// loop unrolled) and fewer LDS round trips:
//   k_colx: a butterfly of each of the pair's columns in registers from the load to the
//           store, four LDS exchanges (forward plan [C0,C1,C2], inverse [C2,C1,C0]).
//   k_rowm: as k_rowx, and the first inverse and last forward stages load and store the block directly, 16
//           elements per thread (1024 x 4 lines, 512 x 4, 256 x 8).
//   k_rowx: the last inverse stage leaves each thread holding whole columns
//           (T = W/F0 threads, columns tid + k*T for all R lines), so rounding,
//           the carry chain, the stairway hand-off and the weighting all run in
//           registers and feed the first forward stage directly
//           (forward plan [F0,F1,F2], inverse plan [F2,F1,F0]).
// LDS bank model (gfx950, 64 banks of 4 bytes, 16-byte accesses, fitted to rocprofv3's
// SQ_LDS_IDX_ACTIVE over probe patterns): a read serves 32 lanes per two cycles, taking as many
// cycles as the most distinct 16-byte slots among them that share a slot index mod 16; a write
// serves 8 lanes per cycle, as many cycles as the most distinct slots sharing an index mod 8.
// LDS is padded by one element per 16 (index i -> i + i/16) so that the strided accesses of the
// FFT stages spread over the banks, and consecutive line (row pass) or column (column pass)
// regions start 6 (row pass, 4 or 8 lines) or 4 elements apart mod 16, which keeps the writes
// that span several regions (the row pass's slot-order scatter, the column pass's first stage)
// on distinct slots mod 8. (8-byte accesses: a write serves 16 lanes per cycle, slots mod 16, a read 32
// lanes, slots mod 32.)
#pragma once

#include <type_traits>

#include "kcommon.h"
#include "coltab.h"

#define CONSTANT __attribute__((address_space(4)))

__device__ __forceinline__ int padi(int i) { return i + (i >> 4); }
// region strides in 16-byte elements (the host sizes LDS with the same formulas)
template<int W, int R> constexpr int rowRegion() { return W + W / 16 + ((R == 4 || R == 8) ? 6 : 4); }
template<int H> constexpr int colRegion() { return H + H / 16 + 4; }

// One LDS -> LDS radix-R autosort stage over NFFT FFTs of length L stored in
// padded regions; Ns is the product of the earlier radices. The twiddle of butterfly input k
// at p = j mod Ns is exp(-2 pi i p*k/(Ns*R)) = tw(p*STRIDE*k) with tw(m) = exp(-2 pi i m/L); the
// provider's st<Ns*R>(p, k, STRIDE) returns it (from a table of the (Ns*R)-th roots when it has one).
// PRIV: the caller allows wave-private stages. A stage with 64 butterflies per FFT
// (or a one-wave group) reads and writes only its own wave's regions; LDS operations of
// one wave complete in order, so such a stage needs no workgroup barrier, only a compiler
// fence. The caller puts a __syncthreads() after the last stage when the next phase
// reads across waves.
template<int L, int T, int R, bool PRIV> constexpr bool stagePrivate() { return PRIV && (T == 64 || L / R == 64); }

template<int L, int REG, int NFFT, int T, bool INV, int R, int Ns, bool PRIV = false, class TW>
__device__ __forceinline__ void xstage(T2* lds, const TW& tw, int tid) {
  constexpr bool priv = stagePrivate<L, T, R, PRIV>();
  constexpr int NB = L / R;
  constexpr int TOT = NB * NFFT;
  constexpr int MB = (TOT + T - 1) / T;
  constexpr int STRIDE = L / (Ns * R);
  T2 v[MB][R];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int g = tid + m * T;
    if (TOT % T == 0 || g < TOT) {
      const int f = g / NB, j = g % NB;
      const T2* x = lds + f * REG;
      if constexpr (NB % 16 == 0) {  // padi(j + k*NB) = padi(j) + k*(NB + NB/16)
        const T2* xj = x + padi(j);
#pragma unroll
        for (int k = 0; k < R; ++k) { v[m][k] = xj[k * (NB + NB / 16)]; }
      } else {
#pragma unroll
        for (int k = 0; k < R; ++k) { v[m][k] = x[padi(j + k * NB)]; }
      }
      if constexpr (Ns > 1) {
        const int p = j % Ns;
#pragma unroll
        for (int k = 1; k < R; ++k) {
          T2 w = tw.template st<Ns * R, R>(p, k, STRIDE);
          v[m][k] = INV ? cmulc(v[m][k], w) : cmul(v[m][k], w);
        }
      }
      Dft<R, INV>::run(v[m]);
    }
  }
  if (priv) {
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int g = tid + m * T;
    if (TOT % T == 0 || g < TOT) {
      const int f = g / NB, j = g % NB;
      T2* x = lds + f * REG;
      const int p = j % Ns;
      const int base = (j - p) * R + p;
      if constexpr (Ns % 16 == 0) {  // padi(base + k*Ns) = padi(base) + k*(Ns + Ns/16)
        T2* xb = x + padi(base);
#pragma unroll
        for (int k = 0; k < R; ++k) { xb[k * (Ns + Ns / 16)] = v[m][k]; }
      } else if constexpr (Ns == 1 && 16 % R == 0) {  // base = j*R: the R outputs stay in one 16-run
        T2* xb = x + padi(base);
#pragma unroll
        for (int k = 0; k < R; ++k) { xb[k] = v[m][k]; }
      } else {
#pragma unroll
        for (int k = 0; k < R; ++k) { x[padi(base + k * Ns)] = v[m][k]; }
      }
    }
  }
  if (priv) {
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

template<int L, int REG, int NFFT, int T, bool INV, bool PRIV, int Ns, int... Rs> struct XStages;
template<int L, int REG, int NFFT, int T, bool INV, bool PRIV, int Ns>
struct XStages<L, REG, NFFT, T, INV, PRIV, Ns> {
  template<class TW> __device__ __forceinline__ static void run(T2*, const TW&, int) {}
};
template<int L, int REG, int NFFT, int T, bool INV, bool PRIV, int Ns, int R, int... Rs>
struct XStages<L, REG, NFFT, T, INV, PRIV, Ns, R, Rs...> {
  template<class TW> __device__ __forceinline__ static void run(T2* lds, const TW& tw, int tid) {
    xstage<L, REG, NFFT, T, INV, R, Ns, PRIV>(lds, tw, tid);
    if constexpr (sizeof...(Rs) > 0) {
      // a workgroup-wide stage after a wave-private one reads what other waves wrote
      constexpr int next[] = {Rs...};
      if constexpr (stagePrivate<L, T, R, PRIV>() && !stagePrivate<L, T, next[0], PRIV>()) { __syncthreads(); }
    }
    XStages<L, REG, NFFT, T, INV, PRIV, Ns * R, Rs...>::run(lds, tw, tid);
  }
};

// exp(-2 pi i m / L) from a table in global memory
struct GlobalTw {
  const T2* t;
  __device__ __forceinline__ T2 operator()(int m) const { return gld(t + m); }
  template<int NR, int RR> __device__ __forceinline__ T2 st(int p, int k, int stride) const { return (*this)(p * stride * k); }
  __device__ __forceinline__ T2 pk(int p, int k) const { return (*this)(p * k); }
};

// Exact product tables for the stages whose twiddles are n-th roots with n = Ns*R small (Ns <= 16
// butterfly phases p, R <= 16): entry (p, k) = w_n^(p*k) for p < P and 1 <= k <= K, one correctly
// rounded value per twiddle instead of the product of two, stored at p*KS + k - 1 with an odd row
// stride KS >= K. The 16 lanes of one LDS access phase read (p, k) for 16 consecutive p and one k:
// 16 entries KS apart, which an odd KS puts in 16 distinct 16-byte bank slots (64 banks). (A table
// of the n-th roots indexed by p*k puts them 2 to 16 in one slot for most k, padded or not.)
// `full` holds w_L^m at m, and w_n = w_L^stride.
template<int P, int K, int KS>
__device__ __forceinline__ void fillProd(const T2* full, int stride, T2* tab, int tid, int T) {
  static_assert(KS % 2 == 1 && KS >= K, "product table stride");
  for (int i = tid; i < P * KS; i += T) {
    const int p = i / KS, k = i % KS + 1;
    tab[i] = k <= K ? gld(full + p * k * stride) : make_double2(0, 0);
  }
}

// The low-part tables TA[i] = w^i (i < 64) below are read at i = (p*k*stride) & 63 for the lanes
// p of a wave and a fixed k; for even k many lanes of one LDS access phase would then hit the same
// banks (k = 8: eight distinct entries i = 0, 8, 16, ... in one bank row of 64 4-byte banks). TA
// is therefore stored with one pad slot after every 16 entries (entry i at i + i/16, 68 slots),
// which spreads those entries over the banks (about half the bank cycles of the unpadded table
// for the row pass's stages, a fifth less for the column pass's).
__device__ __forceinline__ constexpr int taPos(int i) { return i + (i >> 4); }
constexpr int TA_SLOTS = 68;
// table position p of TA (p < TA_SLOTS) -> entry index, -1 for a pad slot
__device__ __forceinline__ constexpr int taEntry(int p) { return (p % 17 == 16) ? -1 : 16 * (p / 17) + p % 17; }

// Row-pass twiddles staged in LDS (ROWTW_SIZE entries after the line regions and the
// round-off slots): w_W^m = TA[m & 63] * TB[m >> 6], TA[i] = w_W^i, TB[j] = w_W^(64 j),
// each twiddle a product of two correctly rounded table entries. Used for W >= 512; at
// W = 256 the fill (68 entries for a 16 KB block) costs more than the global reads save.
// The radix-F1 stages whose twiddles are (F1*F2)-th roots or coarser (the inverse stage before the
// last, Ns = F2, and the second forward stage, Ns = F0 dividing F2) read them from the product
// table of the (F1*F2)-th roots after it (fillProd: F2 rows, stride F1 - 1; at most T = W/F0 =
// F1*F2 slots are reserved): phase p of such a stage reads row p * (F1*F2) / (Ns*F1).
//
// The other twiddles are w_W^(p*k) for a phase p and k < 16 (the last forward stage, Ns*R = W,
// and the last inverse stage, p = tid, k < F0). TA[p*k & 63] for 16 consecutive p hits as few
// as a quarter of the bank slots for odd k; from W = 1024 up they are instead
// P2[(p >> 4) * k] * P1[p & 15][k] with P1[t][k] = w_W^(t*k) (t < 16, k < 16: a product table
// as above, stride 15) and P2[j] = w_W^(16 j) (j < W/16; one entry for the 16 lanes of an access
// phase): again the product of two correctly rounded entries, now without bank conflicts. Layout
// from W = 1024: the (F1*F2)-th-root product table (T slots), P1 (240), P2 (W/16), no TA/TB.
constexpr int ROWTW_SIZE = TA_SLOTS + 64;
template<int W, int T> constexpr int rowTwSlots() { return W >= 1024 ? T + 240 + W / 16 : ROWTW_SIZE + T; }
template<int W, int F1, int F2>
struct RowTw {
  static_assert(F1 % 2 == 0 && F2 * (F1 - 1) <= F1 * F2, "row product table");
  static constexpr bool PK = W >= 1024;
  static constexpr int PT = PK ? 0 : ROWTW_SIZE, P1 = F1 * F2, P2 = F1 * F2 + 240;
  const T2* tab;
  __device__ __forceinline__ T2 operator()(int m) const {
    static_assert(!PK, "no TA/TB table from W = 1024 up");
    return cmul(tab[taPos(m & 63)], tab[TA_SLOTS + (m >> 6)]);
  }
  // w_W^(p*k) for p*k < W and 1 <= k < 16
  __device__ __forceinline__ T2 pk(int p, int k) const {
    if constexpr (PK) {
      return cmul(tab[P2 + (p >> 4) * k], tab[P1 + (p & 15) * 15 + k - 1]);
    } else {
      return (*this)(p * k);
    }
  }
  template<int NR, int RR> __device__ __forceinline__ T2 st(int p, int k, int stride) const {
    if constexpr (RR == F1 && (F1 * F2) % NR == 0) {
      return tab[PT + p * ((F1 * F2) / NR) * (F1 - 1) + k - 1];
    } else if constexpr (NR == W && RR <= 16) {
      return pk(p, k);
    } else {
      return (*this)(p * stride * k);
    }
  }
};
template<int W, int T, int F1, int F2>
__device__ __forceinline__ void fillRowTw(const T2* twRow, T2* tab, int tid) {
  static_assert(W % 64 == 0 && W / 64 <= 64 && W % T == 0, "twiddle table");
  using TW = RowTw<W, F1, F2>;
  if constexpr (TW::PK) {
    fillProd<16, 15, 15>(twRow, 1, tab + TW::P1, tid, T);
    for (int j = tid; j < W / 16; j += T) { tab[TW::P2 + j] = gld(twRow + 16 * j); }
  } else {
    constexpr int N = TA_SLOTS + W / 64;
#pragma unroll
    for (int p = tid; p < N; p += T) {
      const int e = p < TA_SLOTS ? taEntry(p) : 64 * (p - TA_SLOTS);
      tab[p] = e < 0 ? make_double2(0, 0) : gld(twRow + e);
    }
  }
  fillProd<F2, F1 - 1, F1 - 1>(twRow, W / (F1 * F2), tab + TW::PT, tid, T);
}

// Column-pass twiddles staged in LDS after the data regions (colTwSize<H>() entries):
// w_H^m = TA[m & 63] * TB[m >> 6] for m < H, and for column h of the pair the mid
// twiddles w_ND^(a*l) = MA[h][l & 63] * MB[h][l >> 6] and S[h][k] = w_ND^(a*k*H/16).
// Each twiddle is a product of two correctly rounded table entries. Layout: TA (72 slots,
// padded as above), TB[H/64], then per column MA[64], MB[H/64], S[16] (MA is read at
// consecutive l, which needs no padding); sized per H so that small-H groups keep their LDS
// footprint (and so the number of groups per CU) as low as the data allows.
template<int H> constexpr int colTwPer() { return 64 + H / 64 + 16; }
template<int H> constexpr int colTwSize() { return TA_SLOTS + H / 64 + 2 * colTwPer<H>(); }
template<int H>
struct ColTw {
  static_assert(H % 64 == 0 && H / 64 <= 64, "twiddle table");
  static constexpr int MID = TA_SLOTS + H / 64;  // start of column 0's part
  const T2* tab;
  __device__ __forceinline__ T2 operator()(int m) const { return cmul(tab[taPos(m & 63)], tab[TA_SLOTS + (m >> 6)]); }
  template<int NR, int RR> __device__ __forceinline__ T2 st(int p, int k, int stride) const { return (*this)(p * stride * k); }
  __device__ __forceinline__ T2 mid(int h, int l) const {
    const T2* p = tab + MID + h * colTwPer<H>();
    return cmul(p[l & 63], p[64 + (l >> 6)]);
  }
  __device__ __forceinline__ T2 s(int h, int k) const { return tab[MID + h * colTwPer<H>() + 64 + H / 64 + k]; }
};
// Entry i of the twiddle table of the column pair (a0, a1).
template<int H>
__device__ __forceinline__ T2 colTwEntry(const JobDesc& J, int i, int a0, int a1) {
  constexpr int NHI = H / 64, MID = ColTw<H>::MID, PER = colTwPer<H>();
  T2 v;
  if (i < TA_SLOTS) {
    const int e = taEntry(i);
    v = e < 0 ? make_double2(0, 0) : gld(J.twCol + e);
  } else if (i < MID) {
    v = gld(J.twCol + 64 * (i - TA_SLOTS));
  } else {
    const int h = (i - MID) / PER, r = (i - MID) % PER;
    const int a = h ? a1 : a0;
    if (r < 64) {
      v = gld(J.twMidA + a * 64 + r);
    } else if (r < 64 + NHI) {
      v = gld(J.twMidB + a * J.nHi + (r - 64));
    } else {
      v = gld(J.twMidS + a * 16 + (r - 64 - NHI));
    }
  }
  return v;
}
template<int H>
__device__ __forceinline__ void fillColTw(const JobDesc& J, T2* tab, int a0, int a1, int tid, int T) {
  for (int i = tid; i < colTwSize<H>(); i += T) { tab[i] = colTwEntry<H>(J, i, a0, a1); }
}
// ---------------------------------------------------------------- column pass, mirrored pair
// The two columns of a pair have frequencies a and W - a. Transforming the conjugate of column
// W - a takes exactly column a's twiddles (w_ND^(-(W-a)*l) = w_ND^(a*l) * w_H^(-l), and the w_H^(-l)
// only shifts the output index), and its output b is conj(X_{W-a}[H-1-b]): the pairing partner
// of X_a[b], already conjugated. So in a row of 16 lanes the first 8 run butterflies of column a and the
// others the same butterflies of column W - a, with the same twiddles; after the last forward stage a
// lane's partner bins are in the lane 8 away, and the pairing and the first inverse stage run in registers
// (forward plan [C0, C1, C2], inverse [C2, C1, C0]; four LDS exchanges, where transforming both columns stage by
// stage in LDS took six round trips).
// One butterfly per thread. SPLIT: real and imaginary parts are exchanged one after the other through one region
// of doubles per column, in at most 128 VGPRs, so that at H = 3840 two groups and four waves per SIMD share a CU;
// otherwise whole complex elements, with half the barriers.
// LDS positions are sums (one address per butterfly, the rest in the instructions' offsets) and free of
// bank conflicts: rows of a Ns = 1 exchange are odd (C + 1 for even C), the blocks of the others C apart, so
// that consecutive butterflies write distinct slots; the two columns' regions use different halves of the banks
// and alternate by 16 lanes.
// NT: non-temporal loads and stores.
// Measured (HIP events, us per launch, the pass before it in parentheses): 1024 x 3840 split 38.6 (46.1), 1024 x 2560
// split 28.9 (35.4), 1024 x 1536 20.2 (23.4), 256 x 2304 18.9 (20.3), 256 x 512 9.5 (13.5).
// Values derived from i before and after are computed anew instead of being held in registers.
#define FRESH(i) asm volatile("" : "+v"(i))
// Fixes the place of the values in the instruction stream.
template<int N> __device__ __forceinline__ void pin(T2* v) {
#pragma unroll
  for (int k = 0; k < N; ++k) { asm volatile("" : "+v"(v[k].x), "+v"(v[k].y)); }
}
// Element at a 32-bit byte offset from a uniform base: one VGPR of address per access (a state buffer
// is below 4 GiB), where element pointers would hold two.
template<bool NT> __device__ __forceinline__ T2 ldo(const T2* base, uint32_t bytes) {
  return ldx<NT>((const T2*)((const char*)base + bytes));
}
template<bool NT> __device__ __forceinline__ void sto(T2* base, uint32_t bytes, T2 v) { stx<NT>((T2*)((char*)base + bytes), v); }

// f on the part of v that an exchange of elements E moves in round p: v itself, or its real, then its imaginary part
template<class E, class F> __device__ __forceinline__ void part(T2& v, int p, F f) {
  if constexpr (std::is_same_v<E, double>) {
    f(p ? v.y : v.x);
  } else {
    f(v);
  }
}
__device__ __forceinline__ void swapIf(bool c, T2& a, T2& b) {
  const T2 t = a;
  a = make_double2(c ? b.x : a.x, c ? b.y : a.y);
  b = make_double2(c ? t.x : b.x, c ? t.y : b.y);
}
// v of the lane 8 away in the row of 16 (DPP row rotate by 8)
__device__ __forceinline__ double lane8(double v) {
  const uint64_t x = __double_as_longlong(v);
  const uint32_t lo = __builtin_amdgcn_mov_dpp((int)x, 0x128, 0xf, 0xf, true);
  const uint32_t hi = __builtin_amdgcn_mov_dpp((int)(x >> 32), 0x128, 0xf, 0xf, true);
  return __longlong_as_double((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ T2 lane8(T2 v) { return make_double2(lane8(v.x), lane8(v.y)); }

// x[k] *= w^k (conj: by its conjugate) for 1 <= k < C <= 16, w^k exact from load(k): the first six loaded beforehand
// (w), each later one into the registers of the one six before it, which is used up. (Products of loaded powers raised the
// error of a squaring by 1 to 3%.)
template<int C> struct Powers {
  static constexpr int N = C <= 6 ? C - 1 : 6;
  T2 w[N];
  template<typename Load> __device__ __forceinline__ void begin(Load load) {
#pragma unroll
    for (int k = 1; k <= N; ++k) { w[k - 1] = load(k); }
  }
  template<bool CONJ, typename Load> __device__ __forceinline__ void apply(T2* x, Load load) {
#pragma unroll
    for (int k = 1; k < C; ++k) {
      T2& t = w[(k - 1) % N];
      x[k] = CONJ ? cmulc(x[k], t) : cmul(x[k], t);
      pin<1>(&x[k]);
      if (k + N < C) { t = load(k + N); }
    }
  }
};

// Dft<R> with the sub-transforms of a composite R kept one after the other: left to itself the
// scheduler interleaves them, and their temporaries spill.
template<int R> struct Coprime {
  static constexpr int P = 0, Q = 0;
};
template<> struct Coprime<10> { static constexpr int P = 2, Q = 5; };
template<> struct Coprime<14> { static constexpr int P = 2, Q = 7; };
template<> struct Coprime<15> { static constexpr int P = 3, Q = 5; };
template<int R, bool INV> __device__ __forceinline__ void dftSeq(T2* a) {
  constexpr int P = Coprime<R>::P, Q = Coprime<R>::Q;
  pin<R>(a);
  if constexpr (P != 0) {
    T2 b[Q][P];
#pragma unroll
    for (int n2 = 0; n2 < Q; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < P; ++n1) { b[n2][n1] = a[pfaIn<P, Q>(n1, n2)]; }
      Dft<P, INV>::run(b[n2]);
      pin<P>(b[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) {
      T2 c[Q];
#pragma unroll
      for (int n2 = 0; n2 < Q; ++n2) { c[n2] = b[n2][k1]; }
      Dft<Q, INV>::run(c);
      pin<Q>(c);
#pragma unroll
      for (int k2 = 0; k2 < Q; ++k2) { a[pfaOut<P, Q>(k1, k2)] = c[k2]; }
    }
  } else if constexpr (R == 16) {
    T2 b[4][4];
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) {
#pragma unroll
      for (int k1 = 0; k1 < 4; ++k1) { b[k2][k1] = a[4 * k1 + k2]; }
      Dft<4, INV>::run(b[k2]);
#pragma unroll
      for (int m1 = 1; m1 < 4; ++m1) { b[k2][m1] = rootMul<16, INV>(b[k2][m1], k2 * m1); }
      pin<4>(b[k2]);
    }
#pragma unroll
    for (int m1 = 0; m1 < 4; ++m1) {
      T2 c[4];
#pragma unroll
      for (int k2 = 0; k2 < 4; ++k2) { c[k2] = b[k2][m1]; }
      Dft<4, INV>::run(c);
      pin<4>(c);
#pragma unroll
      for (int m2 = 0; m2 < 4; ++m2) { a[m1 + 4 * m2] = c[m2]; }
    }
  } else {
    Dft<R, INV>::run(a);
  }
}

// Grid (W/2, batch), T threads, LDS 2*colRegionX(H) doubles (the two columns) and ColTab::LDS twiddles; modes as k_col
// (SQ: COL_SQUARE only, compiled alone because the other modes' registers would spill in it).
template<int H, int T, int C0, int C1, int C2, bool SPLIT, bool NT, bool SQ>
__global__ __launch_bounds__(T, SPLIT ? 4 : 2) void k_colx(const JobDesc* __restrict__ jobs, int modeArg, int fi, int oi) {
  using L = ColTab<H, C0, C1, C2>;
  static_assert(L::LDS == (int)colTabLds(H) && colRadices(H).c0 == C0 && colRadices(H).c2 == C2, "column table");
  constexpr int REG = colRegionX(H, SPLIT);
  using E = std::conditional_t<SPLIT, double, T2>;
  constexpr int NB0 = H / C0, NB1 = H / C1, NB2 = H / C2, B = T / 2;
  static_assert(C0 * C1 * C2 == H && NB0 <= B && NB1 <= B && NB2 <= B && (NB2 + 31) / 32 == T / 64 && B <= L::ROOTS, "plan");
  constexpr int CM = C0 > C1 ? (C0 > C2 ? C0 : C2) : (C1 > C2 ? C1 : C2);
  const int mode = SQ ? COL_SQUARE : modeArg;
  extern __shared__ T2 lds[];
  T2* const tab = lds + (SPLIT ? 1 : 2) * REG;
  const JobDesc& J = jobs[blockIdx.y];
  const int W = J.W, R = J.R, lgR = J.lgR;
  // XCD x (group i runs on XCD i mod 8) takes the pairs x*W/16 ...: neighbouring pairs share a line
  // block's 256-byte runs, which then go through one L2
  const int q = (blockIdx.x & 7) * (W / 16) + (blockIdx.x >> 3);
  // Column of the pair and butterfly: rows of 16 lanes alternate between the columns; in the middle (last forward,
  // first inverse stage, names ending in P) runs of 8, so that the partner is in the same row.
  const int h = (threadIdx.x >> 4) & 1, hP = (threadIdx.x >> 3) & 1;
  int j = (threadIdx.x >> 5) * 16 + (threadIdx.x & 15), jP = (threadIdx.x >> 4) * 8 + (threadIdx.x & 7);
  E* const reg = reinterpret_cast<E*>(lds) + h * REG;  // the column's region
  E* const regP = reinterpret_cast<E*>(lds) + hP * REG;
  T2* io = J.freq[fi];
  const T2* other = (mode == COL_MUL) ? J.freq[oi] : nullptr;
  const uint32_t WR = (uint32_t)(W * R), colBase = (uint32_t)(2 * q * R);
  // line l of column c lies at element spos(c, l); line j + k*NB0 at spos(h, j) + k*kStride/16 (the host runs this
  // pass only when R divides NB0)
  const uint32_t kStride = (uint32_t)(NB0 >> lgR) * WR * 16;
  auto spos = [&](int c, int l) -> uint32_t {
    return (uint32_t)(l >> lgR) * WR + colBase + (uint32_t)(c << lgR) + (uint32_t)(l & (R - 1));
  };
  // Mid twiddle of line j + k*NB0: base * S[k], the S entries uniform. For q = 0 column 0 has none and column W/2
  // its own; the latter pairs with itself, so it is not conjugated.
  const int a = q ? q : W / 2;
  const double sgn = (q && h) ? -1.0 : 1.0;
  auto midBase = [&](int l) -> T2 { return gld(J.twMidBase + a * NB0 + l); };
  auto mid = [&](T2 base, int k) -> T2 {
    const CONSTANT double* s = (const CONSTANT double*)(J.twMidM + a * 16 + k);
    T2 w = k ? cmul(base, make_double2(s[0], s[1])) : base;
    if (!q) {
      asm volatile("");  // a branch that all other groups skip, not selects in every group
      if (!h) { w = make_double2(1, 0); }
    }
    return w;
  };
  auto root = [&](int t, int k) -> T2 { return gld(J.colTab + L::LDS + t + (k - 1) * L::ROOTS); };  // w_H^(t*k)

  constexpr std::integral_constant<int, C0> c0;
  constexpr std::integral_constant<int, C1> c1;
  constexpr std::integral_constant<int, C2> c2;
  // A stage with NB < T/2 butterflies runs in the waves that have one (uniform branches); the lanes past NB in
  // the last of them repeat butterfly NB - 1 (same addresses, same values).
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto runs = [&](int nb) -> bool { return nb == B || wave < (nb + 31) / 32; };
  auto bf = [&](int nb) -> int { return nb % 32 == 0 ? j : min(j, nb - 1); };
  if (NB2 % 32) { jP = min(jP, NB2 - 1); }

  T2 x[CM];
  // One exchange: nw butterflies write x[k], k < n, at w + k*ws, nr butterflies read x[k], k < m, at r + k*rs; real
  // parts, then imaginary parts.
  auto exchange = [&](auto n, int nw, E* w, int ws, auto m, int nr, const E* r, int rs) {
#pragma unroll
    for (int p = 0; p < (SPLIT ? 2 : 1); ++p) {
      __syncthreads();
      if (runs(nw)) {
#pragma unroll
        for (int k = 0; k < n; ++k) { part<E>(x[k], p, [&](auto& e) { w[k * ws] = e; }); }
      }
      __syncthreads();
      if (runs(nr)) {
#pragma unroll
        for (int k = 0; k < m; ++k) { part<E>(x[k], p, [&](auto& e) { e = r[k * rs]; }); }
      }
    }
  };
  for (int i = threadIdx.x; i < L::LDS; i += T) { tab[i] = gld(J.colTab + i); }
  if (runs(NB0)) {
    const int j0 = bf(NB0);
    const uint32_t o = spos(h, j0) * 16;
#pragma unroll
    for (int k = 0; k < C0; ++k) { x[k] = ldo<NT>(io, o + k * kStride); }
    const T2 base = midBase(j0);
#pragma unroll
    for (int k = 0; k < C0; ++k) {
      x[k] = cmul(make_double2(x[k].x, sgn * x[k].y), mid(base, k));
      pin<1>(&x[k]);
    }
    dftSeq<C0, false>(x);
  }
  FRESH(j);
  // stage 1: radix C1, Ns = C0
  {  // rows of C0 | 1; NB1 is a multiple of C0
    const int j1 = bf(NB1);
    constexpr int PAD = (C0 | 1) - C0;
    exchange(c0, NB0, reg + bf(NB0) * (C0 | 1), 1, c1, NB1, reg + j1 + j1 / C0 * PAD, NB1 + NB1 / C0 * PAD);
  }
  if (runs(NB1)) {
    const T2* t = tab + L::A + (bf(NB1) % C0) * L::KS - 1;
#pragma unroll
    for (int k = 1; k < C1; ++k) {
      x[k] = cmul(x[k], t[k]);
      pin<1>(&x[k]);
    }
    dftSeq<C1, false>(x);
  }
  FRESH(j);
  // stage 2: radix C2, Ns = C0*C1 = NB2: bins j + k*NB2
  Powers<C2> wt;
  wt.begin([&](int k) { return root(jP, k); });
  {  // blocks of C0*C1 = NB2 elements, C0 further apart
    const int j1 = bf(NB1), blk = j1 / C0;
    exchange(c1, NB1, reg + j1 + blk * NB2, C0, c2, NB2, regP + jP, NB2 + C0);
  }
  T2 wb = wt.w[0];
  wt.template apply<false>(x, [&](int k) { return root(jP, k); });
  dftSeq<C2, false>(x);
  pin<C2>(x);
  FRESH(jP);

  if (mode == COL_FWD) {  // the plain spectrum: column W - a's bin H-1-b is conj(x[k])
#pragma unroll
    for (int k = 0; k < C2; ++k) {
      const int b = jP + k * NB2;
      stx<false>(io + spos(hP, q && hP ? H - 1 - b : b), q && hP ? conj2(x[k]) : x[k]);
    }
    return;
  }

  // pairing, with P = conj(partner): X <- X*Y - (1 + w)(X - P)(Y - Q)/4, where Y, Q are the second operand's bins
  // (X, P themselves when squaring); w of bin b is w_ND^(a + W*b). P is in the lane 8 away; for q = 0 columns 0 (b
  // pairs with -b) and W/2 (b with H-1-b) pair within themselves: bin j + k*NB2 with bin (NB2 - j or NB2 - 1 - j) +
  // (C2-1-k)*NB2, through LDS two registers at a time (j = 0 of column 0: bin k*NB2 with (C2-k)*NB2, kept apart).
  wb = cscale(cmul(gld(J.twPair + (q || hP ? a : 0)), wb), 0.25);
  T2* const self = lds + 2 * T;
  if (!q) {
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int k = 0; k < C2; ++k) { self[k] = x[k]; }
    }
  }
#pragma unroll
  for (int k = 0; k < (C2 + 1) / 2; ++k) {
    const int k2 = C2 - 1 - k;
    T2 P, P2;
    if (q) {
      P = lane8(x[k]);
      P2 = lane8(x[k2]);
    } else {
      T2* buf = lds + hP * B;
      __syncthreads();
      buf[jP] = x[k];
      buf[T + jP] = x[k2];
      __syncthreads();
      const int jm = hP ? NB2 - 1 - jP : NB2 - jP;
      const bool own = jm == NB2;
      P = conj2(*(own ? self + (k ? C2 - k : 0) : buf + T + jm));
      P2 = conj2(*(own ? self + (C2 - k2) : buf + jm));
    }
#pragma unroll
    for (int i = 0; i < (k == k2 ? 1 : 2); ++i) {
      const int kk = i ? k2 : k;
      pin<1>(&wb);
      const T2 w = rootMul<C2, false>(wb, kk);
      const T2 v = make_double2(0.25 + w.x, w.y);
      const T2 D = csub(x[kk], i ? P2 : P);
      if (SQ || !other) {
        x[kk] = csub(csqr(x[kk]), cmul(v, csqr(D)));
      } else {
        const int b = jP + kk * NB2;
        T2 Y, Q;
        if (q) {
          Y = gld(other + spos(hP, hP ? H - 1 - b : b));
          if (hP) { Y.y = -Y.y; }
          Q = lane8(Y);
        } else {
          Y = gld(other + spos(hP, b));
          Q = conj2(gld(other + spos(hP, hP ? H - 1 - b : b ? H - b : 0)));
        }
        x[kk] = csub(cmul(x[kk], Y), cmul(v, cmul(D, csub(Y, Q))));
      }
      pin<1>(&x[kk]);
    }
  }
  FRESH(jP);

  // inverse stage 0: radix C2, Ns = 1, butterfly jP: the registers
  dftSeq<C2, true>(x);
  // stage 1: radix C1, Ns = C2
  FRESH(j);
  {  // rows of C2 | 1; NB1 is a multiple of C2
    const int j1 = bf(NB1);
    constexpr int PAD = (C2 | 1) - C2;
    exchange(c2, NB2, regP + jP * (C2 | 1), 1, c1, NB1, reg + j1 + j1 / C2 * PAD, NB1 + NB1 / C2 * PAD);
  }
  if (runs(NB1)) {
    const T2* t = tab + L::B + (bf(NB1) % C2) * L::KS - 1;
#pragma unroll
    for (int k = 1; k < C1; ++k) {
      x[k] = cmulc(x[k], t[k]);
      pin<1>(&x[k]);
    }
    dftSeq<C1, true>(x);
  }
  FRESH(j);
  // stage 2: radix C0, Ns = NB0, then the conjugate mid twiddle and the store
  const int j0 = bf(NB0);
  Powers<C0> wi;
  wi.begin([&](int k) { return root(j0, k); });
  {  // blocks of C1*C2 = NB0 elements, C2 further apart
    const int j1 = bf(NB1), blk = j1 / C2;
    exchange(c1, NB1, reg + j1 + blk * NB0, C2, c0, NB0, reg + j0, NB0 + C2);
  }
  if (runs(NB0)) {
    wi.template apply<true>(x, [&](int k) { return root(j0, k); });
    dftSeq<C0, true>(x);
    pin<C0>(x);
    FRESH(j);
    const T2 base = midBase(bf(NB0));
    const uint32_t o = spos(h, bf(NB0)) * 16;
#pragma unroll
    for (int k = 0; k < C0; ++k) {
      const T2 y = cmulc(x[k], mid(base, k));
      sto<NT>(io, o + k * kStride, make_double2(y.x, sgn * y.y));
    }
  }
}

// ---------------------------------------------------------------- column pass, one region
// The two columns of the pair go through one LDS region in turn, and the real-signal pairing runs in registers: the last
// forward stage (radix C2, T = H/C2 butterflies) leaves thread t holding X0[t + T*k];
// column 1's last stage is computed for butterfly T-1-t, so the partner of X0[b],
// X1[H-1-b], is X1[(T-1-t) + T*(C2-1-k)] in the same thread. The inverse's first stage
// (radix C2, Ns = 1) reads exactly those registers. The pair q = 0 (columns 0 and W/2,
// each paired with itself) goes through LDS. Plan: forward [16, C1, C2], inverse
// [C2, C1, 16]; LDS (colRegion<H>() + colTwSize<H>())*16 bytes, twiddles from the LDS table.
template<int H, int C1, int C2>
__global__ __launch_bounds__(H / C2, 2) void k_coly(const JobDesc* __restrict__ jobs, int mode, int fi, int oi) {
  constexpr int C0 = 16;
  constexpr int T = H / C2;
  constexpr int NB0 = H / C0;
  static_assert(C0 * C1 * C2 == H && T % 64 == 0 && NB0 <= T, "plan");
  constexpr int REG = colRegion<H>();
  extern __shared__ T2 lds[];
  const ColTw<H> tw{lds + REG};
  const JobDesc& J = jobs[blockIdx.y];
  const int W = J.W, R = J.R, lgR = J.lgR;
  const int q = blockIdx.x, tid = threadIdx.x;
  const int a0 = q, a1 = q ? W - q : W / 2;
  T2* io = J.freq[fi];
  const size_t colBase = (size_t)2 * q * R;
  const size_t blockStride = (size_t)W * R;
  auto gpos = [&](int h, int l) -> size_t {
    return (size_t)(l >> lgR) * blockStride + colBase + (h << lgR) + (l & (R - 1));
  };
  const int jl1 = q ? T - 1 - tid : tid;  // column 1's last-stage butterfly
  fillColTw<H>(J, lds + REG, a0, a1, tid, T);
  __syncthreads();

  T2 x0[C2], x1[C2];

  // forward FFT of column h (mid twiddle for column index a), last stage for butterfly jl
  auto forward = [&](int h, int jl, T2* out) {
    if (tid < NB0) {
      const int j = tid;
      const T2 base = tw.mid(h, j);
      T2 v[C0];
#pragma unroll
      for (int k = 0; k < C0; ++k) {
        T2 x = gld(io + gpos(h, j + k * NB0));
        v[k] = cmul(x, k ? cmul(base, tw.s(h, k)) : base);
      }
      Dft<C0, false>::run(v);
#pragma unroll
      for (int k = 0; k < C0; ++k) { lds[padi(j * C0 + k)] = v[k]; }
    }
    __syncthreads();
    XStages<H, REG, 1, T, false, false, C0, C1>::run(lds, tw, tid);
#pragma unroll
    for (int k = 0; k < C2; ++k) { out[k] = lds[padi(jl + k * T)]; }
#pragma unroll
    for (int k = 1; k < C2; ++k) { out[k] = cmul(out[k], tw(jl * k)); }
    Dft<C2, false>::run(out);
    __syncthreads();
  };

  // inverse FFT of column h from registers (butterfly jl of the first stage), then store
  auto inverse = [&](int h, int jl, T2* in) {
    Dft<C2, true>::run(in);
#pragma unroll
    for (int k = 0; k < C2; ++k) { lds[padi(jl * C2 + k)] = in[k]; }
    __syncthreads();
    XStages<H, REG, 1, T, true, false, C2, C1>::run(lds, tw, tid);
    if (tid < NB0) {
      const int j = tid;
      T2 v[C0];
#pragma unroll
      for (int k = 0; k < C0; ++k) { v[k] = lds[padi(j + k * NB0)]; }
#pragma unroll
      for (int k = 1; k < C0; ++k) { v[k] = cmulc(v[k], tw(j * k)); }
      Dft<C0, true>::run(v);
      const T2 base = tw.mid(h, j);
#pragma unroll
      for (int k = 0; k < C0; ++k) {
        gst(io + gpos(h, j + k * NB0), cmulc(v[k], k ? cmul(base, tw.s(h, k)) : base));
      }
    }
    __syncthreads();
  };

  forward(0, tid, x0);
  forward(1, jl1, x1);

  if (mode == COL_FWD) {
#pragma unroll
    for (int k = 0; k < C2; ++k) {
      gst(io + gpos(0, tid + k * T), x0[k]);
      gst(io + gpos(1, jl1 + k * T), x1[k]);
    }
    return;
  }

  const T2* other = (mode == COL_MUL) ? J.freq[oi] : nullptr;
  if (q) {
    const T2 wa = gld(J.twPair + a0);
#pragma unroll
    for (int k = 0; k < C2; ++k) {
      const int b = tid + k * T, bp = H - 1 - b;
      const T2 w = cmul(wa, tw(b));
      if (other) {
        pairMul(x0[k], x1[C2 - 1 - k], gld(other + gpos(0, b)), gld(other + gpos(1, bp)), w);
      } else {
        pairSq(x0[k], x1[C2 - 1 - k], w);
      }
    }
  } else {
    // column 0 pairs b with (H - b) % H, column W/2 pairs b with H - 1 - b
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      T2* x = h ? x1 : x0;
#pragma unroll
      for (int k = 0; k < C2; ++k) { lds[padi(tid + k * T)] = x[k]; }
      __syncthreads();
      const T2 wa = gld(J.twPair + (h ? W / 2 : 0));
      const int last = h ? H / 2 - 1 : H / 2;
      for (int b = tid; b <= last; b += T) {
        const int bp = h ? H - 1 - b : (H - b) % H;
        T2 X = lds[padi(b)], Xp = lds[padi(bp)];
        const T2 w = h ? cmul(wa, tw(b)) : tw(b);
        if (other) {
          pairMul(X, Xp, gld(other + gpos(h, b)), gld(other + gpos(h, bp)), w);
        } else {
          pairSq(X, Xp, w);
        }
        lds[padi(b)] = X;
        if (bp != b) { lds[padi(bp)] = Xp; }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < C2; ++k) { x[k] = lds[padi(tid + k * T)]; }
      __syncthreads();
    }
  }

  inverse(0, tid, x0);
  inverse(1, jl1, x1);
}

// ---------------------------------------------------------------- row pass
// Weight data of one line read through the scalar cache: the line index is uniform across the
// group (readfirstlane), so the loads are scalar and the values live in SGPRs. Vector loads of
// them would also sit in the in-order vector memory counter behind a prefetch still in flight.
struct LineWs {
  double w0, w1, iw0, iw1;
  uint32_t e0, e1;
};
__device__ __forceinline__ LineWs lineWs(const LineW* p) {
  const CONSTANT LineW* q = (const CONSTANT LineW*)p;
  return {q->w[0], q->w[1], q->iw[0], q->iw[1], q->e[0], q->e[1]};
}
// Tagged stairway access through the global address space.
__device__ __forceinline__ uint64_t stairLoad(const uint64_t* p) {
  return __hip_atomic_load((const GLOBAL uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void stairStore(uint64_t* p, uint64_t v) {
  __hip_atomic_store((GLOBAL uint64_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Polls N tagged carries until every tag is current. All N loads are in flight together and a
// round that finds any of them stale reloads all N (a current tag stays current for the rest of
// the launch), so the loop body has no per-carry branches. Bounded: a time-out is flagged to the
// host and the kernel still exits.
template<int N>
__device__ __forceinline__ void pollAll(const JobDesc& J, uint64_t* const* p, uint32_t tag, uint64_t* v) {
#pragma unroll
  for (int k = 0; k < N; ++k) { v[k] = stairLoad(p[k]); }
  for (uint32_t n = 0;; ++n) {
    bool ready = true;
#pragma unroll
    for (int k = 0; k < N; ++k) { ready &= (uint32_t)(v[k] >> 48) == tag; }
    if (ready) { break; }
    if (n >= OWL_SPIN_LIMIT) {
      atomicOr(J.flags + 2, 1u);
      break;
    }
    __builtin_amdgcn_s_sleep(1);
#pragma unroll
    for (int k = 0; k < N; ++k) { v[k] = stairLoad(p[k]); }
  }
}

// What one group of a fused row launch does: block lb; for a first visit (first) only the
// carry-out is published, for a redo (redo) the block is transformed again and nothing is
// published; otherwise it waits for block pred's carries (wrap: the carries of the last block,
// which enter block 0 one column to the right) and publishes its own.
struct FusedItem {
  int lb, pred;
  bool first, redo, wrap, none;
};
// Chunked order (opts bit 4, nb >= 8, grid 8 * (ceil(nb/8) + 1)): group i runs on XCD i mod 8
// (workgroups go to the eight XCDs in turn) and XCD x works through one contiguous chunk of
// blocks B_x .. B_{x+1}-1: its first group visits B_x first (publish only), the next groups take
// the following blocks, and its last group redoes B_{x+1}, the head of the next chunk (block 0
// after the last chunk) once the chunk's last carries are in. Every wait is then on a group of
// the same XCD with a lower index, which that XCD has already started, or on the first group of
// a chunk, which never waits: no start counter is needed. Groups beyond a chunk's items exit.
// Results do not depend on the XCD assignment (any group order gives the same residues); only
// forward progress while kernels of other queues hold parts of the device relies on it.
// Ticket order (otherwise, grid nb + 1): the group's start ticket is its block; ticket nb redoes
// block 0.
// Item of group i of a chunked launch over nb >= 8 blocks (also compiled for the host, where a
// CPU test checks the mapping).
__host__ __device__ inline FusedItem chunkedItem(int nb, int i) {
  FusedItem it{0, 0, false, false, false, false};
  const int x = i & 7, j = i >> 3, q = nb >> 3, rem = nb & 7;
  const int b0 = x * q + (x < rem ? x : rem), c = q + (x < rem ? 1 : 0);
  if (j > c) {
    it.none = true;
  } else if (j == 0) {
    it.lb = b0;
    it.first = true;
  } else if (j < c) {
    it.lb = b0 + j;
    it.pred = it.lb - 1;
  } else {
    const int h = b0 + c;  // the next chunk's head; nb after the last chunk
    it.lb = (h == nb) ? 0 : h;
    it.pred = h - 1;
    it.redo = true;
    it.wrap = h == nb;
  }
  return it;
}
__device__ __forceinline__ FusedItem fusedItem(const JobDesc& J, int opts, int* slot) {
  const int nb = J.nb;
  if (opts & 4) { return chunkedItem(nb, blockIdx.x); }
  FusedItem it{0, 0, false, false, false, false};
  const int g = __builtin_amdgcn_readfirstlane(fusedBlock(J, slot));
  it.lb = (g == nb) ? 0 : g;
  it.pred = g - 1;
  it.first = g == 0;
  it.redo = g == nb;
  it.wrap = g == nb;
  return it;
}

// Pieces of the row pass over one block of R lines, T = W/F0 threads. Thread tid owns columns
// c = tid + k*T (k < F0) of the R lines; v[r][k] holds the inverse transform of (line r,
// column c), then its balanced digits (as doubles), then the weighted digits.
template<int W, int R, int F0, int F1, int F2> struct RowPass {
  static constexpr int T = W / F0;
  static constexpr int LW = R * W;
  static constexpr int NL = LW / T;  // state elements per thread
  static constexpr int REG = rowRegion<W, R>();
  static constexpr bool LDS_TW = W >= 512;
  // k_rowx streams the block with non-temporal accesses from W = 512 up
  static constexpr bool NT = W >= 512;
  using Tw = std::conditional_t<LDS_TW, RowTw<W, F1, F2>, GlobalTw>;

  // Thread tid owns the columns colBase(tid) + k*T (k < F0): colBase permutes the low four bits of
  // tid so that the first forward stage's LDS writes (positions colBase*F0 + k, one per lane) of
  // 8 consecutive lanes fall in 8 distinct bank slots (LDS writes serve 8 lanes per cycle, 16-byte
  // slots mod 8); with colBase = tid they pair up for F0 = 2, 4 and 8. k_row_meta lays out the
  // word metadata with the same permutation.
  __device__ __forceinline__ static int colBase(int tid) {
    const int b = tid & 15, hi = tid & ~15;
    if constexpr (F0 == 2) {
      return hi | (b & 3) | ((b >> 3) << 2) | (((b >> 2) & 1) << 3);
    } else if constexpr (F0 == 4) {
      return hi | (b & 1) | (((b >> 3) & 1) << 1) | (((b >> 1) & 3) << 2);
    } else if constexpr (F0 == 8) {
      return hi | ((b >> 3) & 1) | ((b & 7) << 1);
    } else {
      return tid;
    }
  }

  // element e = s*R + r of the block (slot s, line r) for e = tid + i*T
  __device__ __forceinline__ static void load(const T2* blk, T2* P, int tid) {
#pragma unroll
    for (int i = 0; i < NL; ++i) { P[i] = ldx<NT>(blk + tid + i * T); }
  }
  // ... into the line regions in frequency order
  // LDS position of the block's element e = tid + i*T (slot s = e/R, line r = e%R) in the line
  // regions, frequency order. When T/(2R) is a multiple of 16 the slot of element i is
  // s0 + i*T/R with the same parity as s0, so its frequency moves by +-i*T/(2R) from s0's and its
  // padded position by +-i*(T/(2R))*17/16: one multiply-add per element instead of the division
  // and the slot-to-frequency mapping (the one exception, frequency W/2 in slot 1, is i = 0).
  static constexpr bool LINEAR_SLOTS = T % (2 * R) == 0 && (T / (2 * R)) % 16 == 0;
  struct SlotPos {
    int base, delta, first;
    __device__ __forceinline__ SlotPos(int tid) {
      if constexpr (LINEAR_SLOTS) {
        const int s0 = tid / R, r = tid % R, q0 = s0 >> 1;
        const bool odd = s0 & 1;
        base = r * REG + (odd ? padi(W - q0) : padi(q0));
        delta = (odd ? -1 : 1) * (T / (2 * R)) * 17 / 16;
        first = r * REG + padi(slotFreq(s0, W));
      } else {
        base = delta = first = 0;
      }
    }
    __device__ __forceinline__ int operator()(int tid, int i) const {
      if constexpr (LINEAR_SLOTS) {
        return i == 0 ? first : base + i * delta;
      } else {
        const int e = tid + i * T;
        return (e % R) * REG + padi(slotFreq(e / R, W));
      }
    }
  };
  __device__ __forceinline__ static void scatter(T2* lds, const T2* P, int tid) {
    const SlotPos pos(tid);
#pragma unroll
    for (int i = 0; i < NL; ++i) { lds[pos(tid, i)] = P[i]; }
  }
  // inverse W-point FFT of the R lines (LDS stages, then the radix-F0 stage into registers)
  __device__ __forceinline__ static void inverse(T2* lds, const Tw& tw, int tid, int cb, T2 (&v)[R][F0]) {
    XStages<W, REG, R, T, true, true, 1, F2, F1>::run(lds, tw, tid);
    __syncthreads();
    // last inverse stage (radix F0, Ns = T): butterfly cb of each line -> columns cb + k*T
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int k = 0; k < F0; ++k) { v[r][k] = lds[r * REG + padi(cb + k * T)]; }
#pragma unroll
      for (int k = 1; k < F0; ++k) { v[r][k] = cmulc(v[r][k], tw.pk(cb, k)); }
      Dft<F0, true>::run(v[r]);
    }
  }
  // Unweight, round, carry along the block's 2R words per column. The carry chain runs in
  // FP64: every value is an integer of magnitude below 2^51, so sums, scaling by powers of two
  // and floor are exact. Word u of b bits splits into the carry floor(u/2^b + 1/2) and the
  // balanced digit u - carry*2^b in [-2^(b-1), 2^(b-1)), as the integer chain would.
  // cs[k] = the block's carry-out of column k; roe = max round-off.
  // Word metadata (J.rowMeta, one 64-bit word per thread and block): for the thread's word
  // w = (k*R + r)*2 + rep, bit w says whether it is big (bitsLo + 1 bits) and bit 32 + w whether
  // its weight exponent wrapped (weight halved, inverse weight doubled).
  static_assert(F0 * R * 2 <= 32, "row metadata");
  __device__ __forceinline__ static int bigBit(uint64_t meta, int k, int r, int rep) {
    return (int)((uint32_t)meta >> ((k * R + r) * 2 + rep)) & 1;
  }
  __device__ __forceinline__ static int wrapBit(uint64_t meta, int k, int r, int rep) {
    return (int)((uint32_t)(meta >> 32) >> ((k * R + r) * 2 + rep)) & 1;
  }
  // PIN: line by line in program order (k_rowm, whose registers would spill if lines were interleaved).
  template<bool PIN = false>
  __device__ __forceinline__ static void carry(const JobDesc& J, const LineW* lwBase, const ColW* cw, uint64_t meta,
                                               T2 (&v)[R][F0], double* cs, double& roe, bool llHere, bool mul3) {
#pragma unroll
    for (int k = 0; k < F0; ++k) { cs[k] = 0; }
    const double m3 = mul3 ? 3.0 : 1.0;
    const int bitsLo = J.bitsLo;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const LineWs lw = lineWs(lwBase + r);
#pragma unroll
      for (int k = 0; k < F0; ++k) {
#pragma unroll
        for (int rep = 0; rep < 2; ++rep) {
          const int b = bitsLo + bigBit(meta, k, r, rep);
          const double iw = __builtin_amdgcn_ldexp((rep ? lw.iw1 : lw.iw0) * cw[k].iw, wrapBit(meta, k, r, rep));
          const double x = rep ? v[r][k].y : v[r][k].x;
          const double t = fma(x, iw, OWL_RNDVAL) - OWL_RNDVAL;
          roe = fmax(roe, fabs(fma(x, iw, -t)));
          double u = fma(t, m3, cs[k]);
          if (llHere && r == 0 && k == 0 && rep == 0) { u -= 2; }
          const double c = floor(__builtin_amdgcn_ldexp(u, -b) + 0.5);
          const double dgt = u - __builtin_amdgcn_ldexp(c, b);
          cs[k] = c;
          if (rep) {
            v[r][k].y = dgt;
          } else {
            v[r][k].x = dgt;
          }
        }
        if constexpr (PIN) {
          pin<1>(&v[r][k]);
          asm volatile("" : "+v"(cs[k]), "+v"(roe));
        }
      }
    }
  }
  // Ripples the predecessor's carries through each column's 2R words until they die.
  __device__ __forceinline__ static void ripple(const JobDesc& J, uint64_t meta, T2 (&v)[R][F0], const uint64_t* got) {
    const int bitsLo = J.bitsLo;
#pragma unroll
    for (int k = 0; k < F0; ++k) {
      double carry = (double)unpackCarry(got[k]);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (carry != 0) {
          const int b0 = bitsLo + bigBit(meta, k, r, 0);
          double t = v[r][k].x + carry;
          carry = floor(__builtin_amdgcn_ldexp(t, -b0) + 0.5);
          v[r][k].x = t - __builtin_amdgcn_ldexp(carry, b0);
          if (r == R - 1) {
            v[r][k].y += carry;
            carry = 0;
          } else if (carry != 0) {
            const int b1 = bitsLo + bigBit(meta, k, r, 1);
            t = v[r][k].y + carry;
            carry = floor(__builtin_amdgcn_ldexp(t, -b1) + 0.5);
            v[r][k].y = t - __builtin_amdgcn_ldexp(carry, b1);
          }
        }
      }
    }
  }
  // Weight, then the forward W-point FFT's stage 0 (radix F0, Ns = 1), in registers.
  template<bool PIN = false>
  __device__ __forceinline__ static void weightStage0(const LineW* lwBase, const ColW* cw, uint64_t meta, T2 (&v)[R][F0]) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const LineWs lw = lineWs(lwBase + r);
#pragma unroll
      for (int k = 0; k < F0; ++k) {
        const double w0 = __builtin_amdgcn_ldexp(lw.w0 * cw[k].w, -wrapBit(meta, k, r, 0));
        const double w1 = __builtin_amdgcn_ldexp(lw.w1 * cw[k].w, -wrapBit(meta, k, r, 1));
        v[r][k] = make_double2(v[r][k].x * w0, v[r][k].y * w1);
      }
      Dft<F0, false>::run(v[r]);
      if constexpr (PIN) { pin<F0>(v[r]); }
    }
  }
  // The other forward stages in LDS. The caller has made sure that no thread still reads the
  // line regions.
  __device__ __forceinline__ static void forwardLds(const T2 (&v)[R][F0], T2* lds, const Tw& tw, int tid, int cb) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int k = 0; k < F0; ++k) { lds[r * REG + padi(cb * F0 + k)] = v[r][k]; }
    }
    __syncthreads();
    XStages<W, REG, R, T, false, true, F0, F1, F2>::run(lds, tw, tid);
    __syncthreads();
  }
  // the block from the line regions, slot order
  __device__ __forceinline__ static void store(T2* blk, const T2* lds, int tid) {
    const SlotPos pos(tid);
#pragma unroll
    for (int i = 0; i < NL; ++i) { stx<NT>(blk + tid + i * T, lds[pos(tid, i)]); }
  }
  // the stairway carries this block waits for: block it.pred's, shifted by one column when they
  // wrap around into block 0
  __device__ __forceinline__ static void pollPredecessor(const JobDesc& J, const FusedItem& it, int cb, uint32_t tag,
                                                         uint64_t* got) {
    uint64_t* src[F0];
#pragma unroll
    for (int k = 0; k < F0; ++k) {
      const int c = cb + k * T;
      src[k] = J.stair + (size_t)it.pred * W + (it.wrap ? (c == 0 ? W - 1 : c - 1) : c);
    }
    pollAll<F0>(J, src, tag, got);
    if (it.redo) {  // the block's first visit has read the block before the redo rewrites it
#pragma unroll
      for (int k = 0; k < F0; ++k) { src[k] = J.stair + (size_t)it.lb * W + cb + k * T; }
      uint64_t seen[F0];
      pollAll<F0>(J, src, tag, seen);
    }
  }
  __device__ __forceinline__ static void publish(const JobDesc& J, int g, int cb, uint32_t tag, const double* cs) {
#pragma unroll
    for (int k = 0; k < F0; ++k) { stairStore(J.stair + (size_t)g * W + cb + k * T, packCarry((int64_t)cs[k], tag)); }
  }
};

// Grid (ROW_FUSED: nb + 1, or 8 * (ceil(nb/8) + 1) in chunked order; else nb; batch), T = W/F0
// threads, LDS R*rowRegion<W, R>()*16 + 64
// (+ rowTwSlots<W, T>()*16 for W >= 512) bytes: line regions, per-wave round-off, twiddle tables.
// Modes, options and the tagged stairway as k_row.
template<int W, int R, int F0, int F1, int F2>
__global__ __launch_bounds__(W / F0) void k_rowx(const JobDesc* __restrict__ jobs, int mode, int fi, int wi, int opts,
                                                 uint32_t roeSlot, uint32_t tag) {
  static_assert(F0 * F1 * F2 == W, "plan");
  using P = RowPass<W, R, F0, F1, F2>;
  constexpr int T = P::T, LW = P::LW, REG = P::REG;
  extern __shared__ T2 lds[];
  float* roePart = reinterpret_cast<float*>(lds + R * REG);  // one float per wave, after the line regions
  T2* twTab = lds + R * REG + 4;                               // after the 64 bytes of round-off slots
  const JobDesc& J = jobs[blockIdx.y];
  const typename P::Tw tw{P::LDS_TW ? twTab : J.twRow};
  const int nb = J.nb;
  __shared__ int ticketSlot;
  // the block index is uniform: line weights then come through the scalar cache
  FusedItem it{(int)blockIdx.x, 0, false, false, false, false};
  if (mode == ROW_FUSED) { it = fusedItem(J, opts, &ticketSlot); }
  if (it.none) { return; }
  const int lb = it.lb;
  const int tid = threadIdx.x, cb = P::colBase(tid);
  const bool ll = opts & 1, mul3 = opts & 2;
  T2* blk = J.freq[fi] + (size_t)lb * LW;
  if constexpr (P::LDS_TW) { fillRowTw<W, T, F1, F2>(J.twRow, twTab, tid); }  // read after the first barrier below

  T2 v[R][F0];
  ColW cw[F0];
#pragma unroll
  for (int k = 0; k < F0; ++k) { cw[k] = gld(J.colW + cb + k * T); }
  const uint64_t meta = gld(J.rowMeta + (size_t)lb * T + tid);
  const LineW* lwBase = J.lineW + lb * R;

  if (mode == ROW_LEADIN) {
    const int2* src = J.words[wi] + (size_t)lb * LW;
#pragma unroll
    for (int k = 0; k < F0; ++k) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int2 d = gld(src + (cb + k * T) * R + r);
        v[r][k] = make_double2(d.x, d.y);
      }
    }
  } else {
    {
      T2 x[P::NL];
      P::load(blk, x, tid);
      P::scatter(lds, x, tid);
    }
    __syncthreads();
    P::inverse(lds, tw, tid, cb, v);
    double roe = 0;
    double cs[F0];
    P::carry(J, lwBase, cw, meta, v, cs, roe, ll && lb == 0 && cb == 0, mul3);
    if (mode == ROW_CARRYOUT) {
      roeReport(J, roeSlot, (float)roe);
      int2* dst = J.words[wi] + (size_t)lb * LW;
#pragma unroll
      for (int k = 0; k < F0; ++k) {
        const int c = cb + k * T;
        gst(J.carry[0] + (size_t)lb * W + c, (int64_t)cs[k]);
#pragma unroll
        for (int r = 0; r < R; ++r) { gst(dst + c * R + r, make_int2((int)v[r][k].x, (int)v[r][k].y)); }
      }
      return;
    }
    if (!it.redo) { P::publish(J, lb, cb, tag, cs); }
    if (it.first) {
      roeReport(J, roeSlot, (float)roe);
      return;
    }
    roeWave(roeSlot, (float)roe, roePart);
    uint64_t got[F0];
    P::pollPredecessor(J, it, cb, tag, got);
    P::ripple(J, meta, v, got);
  }
  P::weightStage0(lwBase, cw, meta, v);
  __syncthreads();  // every thread has finished reading the inverse's LDS
  if (mode == ROW_FUSED) { roeGroup(J, roeSlot, roePart, T / 64); }
  P::forwardLds(v, lds, tw, tid, cb);
  P::store(blk, lds, tid);
}

// ---------------------------------------------------------------- row pass, 16 elements per thread
// The same pass as k_rowx with fewer LDS trips, for plans with R*F0 = F2 = 16. The first inverse and
// the last forward stage (radix 16) load and store the block directly: thread (line r, j) holds the
// frequencies j + k*W/16, and with r fastest in a wave every access is R*16 contiguous bytes of one
// slot, while the wave that holds j also holds W/16 - j, whose frequencies lie in the other slots of the
// same lines. Four exchanges go through LDS instead of k_rowx's six trips. SPLIT: real and imaginary parts
// are exchanged one after the other (half the LDS) in at most 128 VGPRs, at 1024 x 4 four groups and
// four waves per SIMD on a CU; otherwise complex elements and half the barriers, two waves per SIMD.
// NT: non-temporal loads and stores; with 4 lines the lanes of j and W/16 - j then trade registers so that one
// access covers whole 128-byte lines (64-byte halves cost a quarter of the non-temporal bandwidth: 25 against 21 us
// for the bare copy of 63 MB; with plain accesses they cost nothing).
// Twiddles: product tables of exact entries in LDS for the middle stages, exact entries of the full
// table for the others (Powers).
// LDS positions are sums without bank conflicts on the writes: exchanges 1 and 3 (Ns = 1) pad one slot per 16,
// exchange 4's blocks are F0 slots further apart; the line strides differ so that lanes of R lines at one
// position do not meet.
// Measured (HIP events, us per fused launch, k_rowx in parentheses): 1024 x 3840 split 38.0 (43.4), 1024 x 1536 complex
// 23.2 (24.2), 64 jobs of 256 x 2304 split 277 (340). Two-line blocks stay with k_rowx, which has more waves for them:
// 512 x 1152 15.7 (18.1 with 16 elements per thread), 1024 x 1408 20.8 (22.7).
template<int W, int R, int F0, int F1, bool SPLIT> struct RowM {
  static constexpr int T = W / F0, J = W / 16, F2 = 16, MB = 16 / F1, NB1 = W / F1;
  static_assert(F0 * F1 * F2 == W && R * F0 == 16 && T % 64 == 0 && NB1 % 16 == 0 && J % 16 == 0, "plan");
  static constexpr RowLayout G = rowLayout(W, R, F0, F1, SPLIT);
  static constexpr int L1 = G.l1, L2 = W, L3 = G.l3, L4 = G.l4;  // line strides of the exchanges, in elements
  static constexpr int KS = G.ks, TAB = G.tab, SLOTS = G.slots;
  // thread's line and butterfly in the first and last stage
  __device__ __forceinline__ static int line(int tid) { return tid % R; }
  __device__ __forceinline__ static int bfly(int tid) {
    constexpr int U = 64 / R;
    const int w = tid >> 6, i = (tid & 63) / R;
    const int lo = w * (U / 2) + i, hi = w * (U / 2) + i - U / 2;
    return i < U / 2 ? lo : hi ? J - hi : J / 2;
  }
  // byte offset of frequency j + k*J of line r within the block
  __device__ __forceinline__ static uint32_t slotOf(int j, int k, int r) {
    const int f = j + k * J;
    const int s = k < 8 ? 2 * f : (k == 8 && f == W / 2) ? 1 : 2 * (W - f) + 1;
    return (uint32_t)(s * R + r) * 16;
  }
};

template<int W, int R, int F0, int F1, bool SPLIT, bool NT, bool FUSED>
__global__ __launch_bounds__(W / F0, SPLIT ? 4 : 2) void k_rowm(const JobDesc* __restrict__ jobs, int modeArg, int fi, int wi, int opts,
                                                    uint32_t roeSlot, uint32_t tag) {
  using M = RowM<W, R, F0, F1, SPLIT>;
  using P = RowPass<W, R, F0, F1, 16>;
  constexpr bool FULL = NT && R == 4;
  constexpr int T = M::T, J_ = M::J, MB = M::MB, NB1 = M::NB1, LW = R * W;
  const int mode = FUSED ? ROW_FUSED : modeArg;
  extern __shared__ T2 lds[];
  using E = std::conditional_t<SPLIT, double, T2>;
  E* const buf = reinterpret_cast<E*>(lds);
  T2* const tab = lds + M::TAB;
  float* const roePart = reinterpret_cast<float*>(lds + M::SLOTS - 4);
  const JobDesc& J = jobs[blockIdx.y];
  const int nb = J.nb;
  __shared__ int ticketSlot;
  FusedItem it{(int)blockIdx.x, 0, false, false, false, false};
  if (mode == ROW_FUSED) { it = fusedItem(J, opts, &ticketSlot); }
  if (it.none) { return; }
  const int lb = it.lb;
  const bool ll = opts & 1, mul3 = opts & 2;
  int tid = threadIdx.x;
  T2* blk = J.freq[fi] + (size_t)lb * LW;

  T2 x[16];
  // Exchange: w(m) and r(m) are the LDS addresses of the thread's butterfly m on either side.
  auto exchange = [&](auto nw, auto mw, auto w, int ws, auto nr, auto mr, auto r, int rs) {
#pragma unroll
    for (int p = 0; p < (SPLIT ? 2 : 1); ++p) {
      __syncthreads();
#pragma unroll
      for (int m = 0; m < mw; ++m) {
        E* d = buf + w(m);
#pragma unroll
        for (int k = 0; k < nw; ++k) { part<E>(x[m * nw + k], p, [&](auto& e) { d[k * ws] = e; }); }
      }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < mr; ++m) {
        const E* d = buf + r(m);
#pragma unroll
        for (int k = 0; k < nr; ++k) { part<E>(x[m * nr + k], p, [&](auto& e) { e = d[k * rs]; }); }
      }
    }
  };
  constexpr std::integral_constant<int, 1> c1;
  constexpr std::integral_constant<int, 16> c16;
  constexpr std::integral_constant<int, F0> cF0;
  constexpr std::integral_constant<int, F1> cF1;
  constexpr std::integral_constant<int, MB> cMB;
  constexpr std::integral_constant<int, R> cR;
  // middle-stage butterfly m of the thread: line and index
  auto line1 = [&](int m) { return (tid + m * T) / NB1; };
  auto bfly1 = [&](int m) { return (tid + m * T) % NB1; };

  if (mode == ROW_LEADIN) {
    fillProd<16, F1 - 1, M::KS>(J.twRow, F0, tab, tid, T);
    const int2* src = J.words[wi] + (size_t)lb * LW;
#pragma unroll
    for (int k = 0; k < F0; ++k) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int2 d = gld(src + (tid + k * T) * R + r);
        x[r * F0 + k] = make_double2(d.x, d.y);
      }
    }
  } else {
    {
      const int r = M::line(tid), j = M::bfly(tid);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t o = M::slotOf(j, k, r), o2 = M::slotOf(j, 15 - k, r);
        const bool up = FULL && (tid & 32);
        x[k] = ldo<NT>(blk, up ? o2 : o);
        x[15 - k] = ldo<NT>(blk, up ? o : o2);
      }
      if constexpr (FULL) {
#pragma unroll
        for (int k = 0; k < 8; ++k) { swapIf(tid & 32, x[k], x[15 - k]); }
      }
    }
    fillProd<16, F1 - 1, M::KS>(J.twRow, F0, tab, tid, T);
    dftSeq<16, true>(x);
    pin<16>(x);
    FRESH(tid);
    // inverse stage 1: radix F1, Ns = 16
    exchange(c16, c1, [&](int) { return M::line(tid) * M::L1 + M::bfly(tid) * 17; }, 1, cF1, cMB,
             [&](int m) { return line1(m) * M::L1 + bfly1(m) + (bfly1(m) >> 4); }, NB1 / 16 * 17);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const T2* t = tab + (bfly1(m) & 15) * M::KS - 1;
#pragma unroll
      for (int k = 1; k < F1; ++k) {
        x[m * F1 + k] = cmulc(x[m * F1 + k], t[k]);
        pin<1>(&x[m * F1 + k]);
      }
      dftSeq<F1, true>(x + m * F1);
      pin<F1>(x + m * F1);
    }
    FRESH(tid);
    // inverse stage 2: radix F0, Ns = T: columns tid + k*T of the R lines
    exchange(cF1, cMB, [&](int m) { return line1(m) * M::L2 + (bfly1(m) & ~15) * F1 + (bfly1(m) & 15); }, 16, cF0, cR,
             [&](int m) { return m * M::L2 + tid; }, T);
    T2 w[F0];
#pragma unroll
    for (int k = 1; k < F0; ++k) { w[k] = gld(J.twRow + tid * k); }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int k = 1; k < F0; ++k) { x[r * F0 + k] = cmulc(x[r * F0 + k], w[k]); }
      Dft<F0, true>::run(x + r * F0);
      pin<F0>(x + r * F0);
    }
    FRESH(tid);
  }

  const uint64_t meta = gld(J.rowMeta + (size_t)lb * T + tid);
  const LineW* lwBase = J.lineW + lb * R;
  T2 (&v)[R][F0] = reinterpret_cast<T2 (&)[R][F0]>(x);
  if (mode != ROW_LEADIN) {
    double roe = 0;
    double cs[F0];
    {
      ColW cw[F0];
#pragma unroll
      for (int k = 0; k < F0; ++k) { cw[k].iw = ((const GLOBAL ColW*)(J.colW + tid + k * T))->iw; }
      P::template carry<true>(J, lwBase, cw, meta, v, cs, roe, ll && lb == 0 && tid == 0, mul3);
    }
    if (mode == ROW_CARRYOUT) {
      roeReport(J, roeSlot, (float)roe);
      int2* dst = J.words[wi] + (size_t)lb * LW;
#pragma unroll
      for (int k = 0; k < F0; ++k) {
        const int c = tid + k * T;
        gst(J.carry[0] + (size_t)lb * W + c, (int64_t)cs[k]);
#pragma unroll
        for (int r = 0; r < R; ++r) { gst(dst + c * R + r, make_int2((int)v[r][k].x, (int)v[r][k].y)); }
      }
      return;
    }
    if (!it.redo) { P::publish(J, lb, tid, tag, cs); }
    if (it.first) {
      roeReport(J, roeSlot, (float)roe);
      return;
    }
    roeWave(roeSlot, (float)roe, roePart);
    uint64_t got[F0];
    P::pollPredecessor(J, it, tid, tag, got);
    P::ripple(J, meta, v, got);
  }
  {
    FRESH(tid);
    ColW cw[F0];
#pragma unroll
    for (int k = 0; k < F0; ++k) { cw[k].w = ((const GLOBAL ColW*)(J.colW + tid + k * T))->w; }
    P::template weightStage0<true>(lwBase, cw, meta, v);
  }
  pin<16>(x);
  // forward stage 1: radix F1, Ns = F0
  exchange(cF0, cR, [&](int m) { return m * M::L3 + tid * F0 + (tid * F0 >> 4); }, 1, cF1, cMB,
           [&](int m) { return line1(m) * M::L3 + bfly1(m) + (bfly1(m) >> 4); }, NB1 / 16 * 17);
  if (mode == ROW_FUSED) { roeGroup(J, roeSlot, roePart, T / 64); }
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const T2* t = tab + (bfly1(m) % F0) * (16 / F0) * M::KS - 1;
#pragma unroll
    for (int k = 1; k < F1; ++k) {
      x[m * F1 + k] = cmul(x[m * F1 + k], t[k]);
      pin<1>(&x[m * F1 + k]);
    }
    dftSeq<F1, false>(x + m * F1);
    pin<F1>(x + m * F1);
  }
  FRESH(tid);
  // forward stage 2: radix 16, Ns = J, then the store
  Powers<16> wt;
  wt.begin([&](int k) { return gld(J.twRow + k * M::bfly(tid)); });
  exchange(cF1, cMB, [&](int m) { return line1(m) * M::L4 + bfly1(m) + bfly1(m) / F0 * J_; }, F0, c16, c1,
           [&](int) { return M::line(tid) * M::L4 + M::bfly(tid); }, J_ + F0);
  wt.template apply<false>(x, [&](int k) { return gld(J.twRow + k * M::bfly(tid)); });
  dftSeq<16, false>(x);
  pin<16>(x);
  FRESH(tid);
  {
    const int r = M::line(tid), j = M::bfly(tid);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t o = M::slotOf(j, k, r), o2 = M::slotOf(j, 15 - k, r);
      const bool up = FULL && (tid & 32);
      if constexpr (FULL) { swapIf(tid & 32, x[k], x[15 - k]); }
      sto<NT>(blk, up ? o2 : o, x[k]);
      sto<NT>(blk, up ? o : o2, x[15 - k]);
    }
  }
}

// ---------------------------------------------------------------- name tables
struct OwlKernelEntry {
  const char* name;
  const void* fn;
  unsigned maxThreads;
};
