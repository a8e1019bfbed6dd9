// Streaming solve of lines from their records.
//
// A workgroup of four waves runs two chains of block rows in lockstep: the
// two halves of a twisted line (TW: chain 0 rows 0..h+1 top-down, chain 1 rows
// n-1..h+2 bottom-up) or two plain lines.  Wave 0 runs the recurrences
//   y_i = c_i + W2_i y_{i-1} + W1_i y_{i-2}
// (forward W2 = N2, W1 = N1, c = Linv b; backward W2 = Q4, W1 = Q5, c = Uinv y);
// wave 1 copies the records into a ring of LDS buffers, waves 2 and 3 form c
// and write the results out.
//
// What bounds it.  Up to about 256 lines the chain: a step is ten
// multiply-adds, two swaps and eight LDS accesses of one wave, 80 ns measured
// (1025 rows, 33 lines: 100 us for 1026 steps, of it 88 without the
// loaders; the earlier form, five broadcasts and four sums over the wave per
// step, took 190 ns).  With more lines the memory: 256 lines of 1025 rows take
// 117 us, 4.9 TB/s of 6.1 that reading alone reaches, and 1024 of 257 rows
// 101 us, 5.6 TB/s; 20 us of that are the results' stores.  A workgroup more
// than a multiple of 256 costs a share of the chip: one CU then streams twice
// as much at the same share of the bandwidth (257 lines of 1025 rows 145 us,
// 1025 of 257 120 us).
//
// Before, with one wave on the recurrence and three that each copied, waited
// and prepared (us, complex double): 257 lines of 1025 rows 208 -> 145, 1025
// of 257 147 -> 120 (twisted) and 133 (plain), 257 of 513 111 -> 72, 65 of 129
// 27 -> 19; complex float 257 of 1025 141 -> 86, 1025 of 257 83 -> 74.
#pragma once
#include "common.hpp"

namespace lns3d {

typedef __attribute__((address_space(3))) void lds_void;

// A lane's share of a block-row product.  In a 16-lane row, lanes 0-4 hold the
// real parts of the five components and lanes 5-9 the imaginary parts, of the
// vector v and of the product.  With a = (re | im) and b = (im | re) of the
// lane's block row by lane group, x += sum_q a_q v_re,q and y = sum_q b_q
// v_im,q, the product's parts are x - y on lanes 0-4 and x + y on lanes 5-9.
// The broadcast of v_q is the DPP operand of the multiply-add itself
// (row_newbcast), so it costs no instruction.  The leading s_nop covers the
// two wait states a DPP read needs after a VALU write of the same register.
#define LNS3D_MAC(SUF, Q, Q5, A, B)                                                   \
  "v_fmac_" SUF "_dpp %0, %2, %" A " row_newbcast:" Q " row_mask:0xf bank_mask:0xf\n" \
  "v_fmac_" SUF "_dpp %1, %2, %" B " row_newbcast:" Q5 " row_mask:0xf bank_mask:0xf\n"
#define LNS3D_MAC5(SUF)                                                                      \
  asm("s_nop 1\n" LNS3D_MAC(SUF, "0", "5", "3", "8") LNS3D_MAC(SUF, "1", "6", "4", "9")      \
          LNS3D_MAC(SUF, "2", "7", "5", "10") LNS3D_MAC(SUF, "3", "8", "6", "11")            \
              LNS3D_MAC(SUF, "4", "9", "7", "12")                                            \
      : "+&v"(x), "+&v"(y)                                                                   \
      : "v"(v), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(b[0]), "v"(b[1]), \
        "v"(b[2]), "v"(b[3]), "v"(b[4]))
__device__ __forceinline__ void row_mac5(double &x, double &y, double v, const double (&a)[5], const double (&b)[5]) {
  LNS3D_MAC5("f64");
}
__device__ __forceinline__ void row_mac5(float &x, float &y, float v, const float (&a)[5], const float (&b)[5]) {
  LNS3D_MAC5("f32");
}
#undef LNS3D_MAC5
#undef LNS3D_MAC

// One step's hand-over between the wave's halves.  p holds partial sums (the
// lower half W2 y_{i-1} + c, the upper half W1 y_{i-2}), v the values they
// were formed from (lower y_{i-1}, upper y_{i-2}).  v_permlane32_swap of p
// with v exchanges p's upper half for v's lower one, after which p holds
// (lower partial sum, y_{i-1}) and v (upper partial sum, y_{i-2}); with low =
// 1 in the lower half and 0 in the upper, p + low v is the next step's v:
// y_i below, y_{i-1} above.  The s_nop covers the wait states the swap needs
// after a VALU write.
__device__ __forceinline__ double hand_over(double p, double v, double low) {
  const unsigned long long pb = __builtin_bit_cast(unsigned long long, p), vb = __builtin_bit_cast(unsigned long long, v);
  unsigned p0 = (unsigned)pb, p1 = (unsigned)(pb >> 32), v0 = (unsigned)vb, v1 = (unsigned)(vb >> 32);
  asm("s_nop 1\n"
      "v_permlane32_swap_b32 %0, %2\n"
      "v_permlane32_swap_b32 %1, %3\n"
      : "+v"(p0), "+v"(p1), "+v"(v0), "+v"(v1));
  return fma(__builtin_bit_cast(double, ((unsigned long long)v1 << 32) | v0), low,
             __builtin_bit_cast(double, ((unsigned long long)p1 << 32) | p0));
}
__device__ __forceinline__ float hand_over(float p, float v, float low) {
  unsigned p0 = __builtin_bit_cast(unsigned, p), v0 = __builtin_bit_cast(unsigned, v);
  asm("s_nop 1\n"
      "v_permlane32_swap_b32 %0, %1\n"
      : "+v"(p0), "+v"(v0));
  return fmaf(__builtin_bit_cast(float, v0), low, __builtin_bit_cast(float, p0));
}

// where a record keeps the two blocks of the recurrence: component m's rows
// of W2 and W1 are 20 reals at 20 m, ten real parts and then ten imaginary
// parts, the columns in the order W2 0 1, W1 0 1, W2 2 3, W1 2 3, W2 4, W1 4.
// A lane of the recurrence reads its half's five parts as two pairs and one
// real, at an offset that depends on the half only.
__host__ __device__ constexpr int rec_pos(int older, int q) {
  return q < 4 ? (q / 2) * 4 + 2 * older + (q & 1) : 8 + older;
}

// the cache policy of the records' copies: non-temporal, as each record is
// read once per solve and the right-hand sides should stay in the L2 beside
// them (256 lines of 1025 rows 124 -> 114 us)
constexpr int NT = 2;

template <int U> using idx_t = std::integral_constant<int, U>;
template <int N, int U = 0, typename F> __device__ __forceinline__ void static_for(F &&f) {
  if constexpr (U < N) {
    f(idx_t<U>());
    static_for<N, U + 1>(f);
  }
}

// T: record precision; R: rows of a chunk (a multiple of three); NBUF: LDS
// buffers; TW: twisted lines, one per workgroup, else two plain lines; RES:
// the lines' right-hand sides stay in LDS from the first row to the last.
//
// The right-hand sides are read from `in` and the solutions left in rhs, of the
// same layout (in == rhs: in place; non-resident lines pass through rhs); a
// refined step's first solve reads the residual so, which was copied before
// (a step of 257x129 142 -> 138 us with the residual formed in the operator's
// kernel, 1025x257 527 -> 517).
//
// PER: periodic lines (plain pairs).  Their bordered LU has the same band, so
// rows 0 .. n-3 are a chain without boundary blocks; the last two rows meet
// every other one:
//   p2[row i]: what y_i adds to rows n-2 and n-1, summed by the waves that
//     otherwise only write out, from the results in LDS;
//   qp[row i]: what x_{n-2} and x_{n-1} add to row i, added where Uinv y is
//     formed.
// They ride through a ring of their own, whose buffers live as long as the
// staged right-hand sides.  Between the passes one
// wave solves rows n-2 and n-1 of both lines.  Bound by the memory from about
// 400 lines (512 lines of 1023 rows, 3760 bytes a row: 382 us, 5.2 TB/s), by
// the waves that prepare and sum below (97 of 256 rows 64 us, 0.76 us a chunk
// where the chain takes 0.48).  Before, one line or four per workgroup, its
// recurrence by broadcasts and the border blocks read from memory where they
// were used: 474 and 92 us.  Border blocks held in registers two chunks ahead
// were slower (473 and 99): the compiler copies them once loaded, and waits.
template <typename T, int R, int NBUF, bool TW, bool RES, bool PER = false> struct LineSolve {
  static_assert(!(TW && PER), "periodic lines are plain");
  static_assert(R % 3 == 0, "three rotating register sets");
  static_assert(NBUF >= 4, "a chunk computed, one being prepared, two in flight");
  static constexpr int NROW = NBUF + 2;      // staged right-hand sides: two chunks more until they are copied out
  // LDS layout in bytes
  static constexpr unsigned CS = sizeof(cx<T>);
  static constexpr unsigned CHB = R * 66 * CS, BUFB = 2 * CHB;   // a chunk's records: one chain, both
  // boundary blocks of a pass; PER: of both lines, the records of rows n-2
  // (60 and 66 values) and n-1 (60, and 16 without its recurrence), their right-hand sides (80 bytes a
  // row), the border sums (20 values) and the waves' shares of them
  static constexpr unsigned TAIL = NBUF * BUFB, BREC = 2 * 202 * CS, BSUM = BREC + 4 * 80, BPART = BSUM + 20 * CS,
                            TAILB = PER ? (BPART + 400 * CS + 15) & ~15u : (150 * CS + 15) & ~15u;
  static constexpr unsigned SV = TAIL + TAILB, SVB = (20 * CS + 15) & ~15u;       // rows kept for them
  static constexpr unsigned ROWB = 80;                           // a right-hand-side row
  static constexpr unsigned ZERO = SV + SVB, DUMMY = ZERO + R * ROWB;
  static constexpr unsigned BORD = DUMMY + R * ROWB, BORDB = PER ? R * 50 * CS : 0;    // PER: a chunk's p2 or qp of one chain
  static constexpr unsigned ROWS = BORD + NROW * 2 * BORDB;      // right-hand-side rows
  // rows of a resident right-hand side: a twisted line's inactive steps
  // touch one row before chain 1 and three after it
  static __host__ __device__ unsigned rows(int n) { return RES ? (TW ? n + 4 : PER ? 2 * (n - 2) : 2 * n) : NROW * 2 * R; }
  static __host__ __device__ unsigned lds_bytes(int n) { return ROWS + rows(n) * ROWB; }

  static __device__ __forceinline__ void run(char *sm, long bid, int n, int h, long L, const cx<T> *__restrict__ fwd,
                                             const cx<T> *__restrict__ bwd, const cx<T> *__restrict__ tail,
                                             const double2 *in, double2 *rhs, long sL, long sR,
                                             const cx<T> *__restrict__ p2 = nullptr,
                                             const cx<T> *__restrict__ qp = nullptr) {
    // rows of a line in memory; of its chain (PER: without the last two)
    const int nmem = n;
    if (PER) n -= 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int len0 = TW ? h + 2 : n, len1 = TW ? n - h - 2 : n;
    // by chain, in arithmetic form: a select here becomes a per-lane table
    // in scratch, whose loads would wait on the copies in flight
    auto len = [&](int c) { return len0 + c * (len1 - len0); };
    auto jtop = [&](int c) { return TW ? len0 - 1 + c * (len1 + 2 - len0) : n - 1; };   // first backward row
    auto line_of = [&](int c) { return TW ? bid : min(2 * bid + c, L - 1); };
    auto real_row = [&](int c, int j) { return TW ? j + c * (n - 1 - 2 * j) : j; };
    const int N = (len0 + R - 1) / R;                  // chunks of a pass
    // Chunk k: LDS slot u holds chain row first_row + u where that exists;
    // step s of the pass is slot s - kR forward, R - 1 - (s - kR) backward.
    auto first_row = [&](bool fw, int k, int c) { return fw ? k * R : jtop(c) - k * R - R + 1; };
    auto row_off = [&](int rb, int c, int jb) -> unsigned {     // slot 0 of a chunk's right-hand sides (rb: its staging buffer)
      if (RES) return ROWS + (unsigned)(c * (TW ? len0 + 1 : n) + jb) * ROWB;
      return ROWS + (unsigned)((rb * 2 + c) * R) * ROWB;
    };

    if (wave != 0) {
      // ---- loader waves ----
      const int w = wave - 1;
      // A round handles 12 rows of a chunk, five lanes a row: this lane's
      // chain c, slot u, chain row j and component
      constexpr int ROUNDS = (2 * R + 11) / 12;
      const int l5 = lane / 5, lq = lane - 5 * l5;
      auto my_row = [&](bool fw, int k, int rnd, int &c, int &u, int &j) {
        const int rr = rnd * 12 + l5;
        c = rr / R;
        u = rr % R;
        j = first_row(fw, k, c) + u;
        return lane < 60 && rr < 2 * R && j >= 0 && j < len(c);
      };
      const long to_in = reinterpret_cast<const char *>(in) - reinterpret_cast<const char *>(rhs);   // no select: see above
      auto value_of = [&](auto *v, int c, int j) { return v + (line_of(c) * sL + (long)real_row(c, j) * sR) * 5 + lq; };
      auto issue = [&](bool fw, int k, int buf, int rb) {
        auto records = [&](auto FWT) {
          constexpr int ROW = (decltype(FWT)::value ? 60 : 66) * CS, FULL = R * ROW;   // bytes of a row, a chunk
          static_assert(FULL >= 1024 && FULL % 16 == 0, "whole copies of 1 KB, the last one overlapping");
#pragma unroll
          for (int c = 0; c < 2; c++) {
            const int jb = first_row(fw, k, c), a = max(0, -jb), b = min(R, len(c) - jb);
            const char *src = reinterpret_cast<const char *>(fw ? fwd : bwd) +
                              (line_of(c) * nmem + (TW ? c * len0 : 0) + jb) * ROW + lane * 16;
            char *dst = sm + (buf * BUFB + c * CHB);
            if (a == 0 && b == R) {
              // 1 KB an instruction (16 B a lane); the last one ends with the
              // chunk and copies some bytes a second time
              static_for<(FULL + 1023) / 1024>([&](auto I) {
                constexpr int at = decltype(I)::value * 1024 + 1024 <= FULL ? decltype(I)::value * 1024 : FULL - 1024;
                constexpr int base = at & ~4095;
                __builtin_amdgcn_global_load_lds((const void *)(src + base), (lds_void *)(dst + base), 16, at - base, NT);
              });
            } else {
              for (int o = a * ROW; o < b * ROW; o += 1024)
                if (o + lane * 16 < b * ROW)
                  __builtin_amdgcn_global_load_lds((const void *)(src + o), (lds_void *)(dst + o), 16, 0, NT);
            }
          }
        };
        if (fw) records(std::true_type{});
        else records(std::false_type{});
        if constexpr (PER) {
          constexpr int ROW = 50 * CS, FULL = R * ROW;
          static_assert(FULL >= 1024 && FULL % 16 == 0, "as the records");
#pragma unroll
          for (int c = 0; c < 2; c++) {
            const int jb = first_row(fw, k, c), a = max(0, -jb), b = min(R, len(c) - jb);
            const char *src = reinterpret_cast<const char *>(fw ? p2 : qp) + (line_of(c) * nmem + jb) * ROW + lane * 16;
            char *dst = sm + (BORD + (rb * 2 + c) * BORDB);
            if (a == 0 && b == R) {
              static_for<(FULL + 1023) / 1024>([&](auto I) {
                constexpr int at = decltype(I)::value * 1024 + 1024 <= FULL ? decltype(I)::value * 1024 : FULL - 1024;
                constexpr int base = at & ~4095;
                __builtin_amdgcn_global_load_lds((const void *)(src + base), (lds_void *)(dst + base), 16, at - base, NT);
              });
            } else {
              for (int o = a * ROW; o < b * ROW; o += 1024)
                if (o + lane * 16 < b * ROW)
                  __builtin_amdgcn_global_load_lds((const void *)(src + o), (lds_void *)(dst + o), 16, 0, NT);
            }
          }
        }
        if (!RES) {
#pragma unroll
          for (int rnd = 0; rnd < ROUNDS; rnd++) {
            int c, u, j;
            if (my_row(fw, k, rnd, c, u, j))
              __builtin_amdgcn_global_load_lds((const void *)(reinterpret_cast<const char *>(value_of(rhs, c, j)) + to_in * fw),
                                               (lds_void *)(sm + (ROWS + rb * 2 * R * ROWB + rnd * 960)), 16, 0, 0);
          }
        }
      };
      auto load_rhs = [&](int part, int parts) {       // RES: the whole right-hand sides
#pragma unroll
        for (int c = 0; c < 2; c++)
          for (int b = part; b * 12 < len(c); b += parts) {
            const int j = b * 12 + l5;
            if (lane < 60 && j < len(c))
              __builtin_amdgcn_global_load_lds((const void *)value_of(in, c, j), (lds_void *)(sm + (row_off(0, c, 0) + b * 960)),
                                               16, 0, 0);
          }
      };
      auto load_tail = [&](bool fw) {                  // boundary blocks of a pass
        if constexpr (PER) {
          if (!fw) return;                             // both passes' at the start
          cx<T> v[7];
          const int e20 = min(lane, 19);
          const double2 b = in[(line_of(e20 / 10) * sL + (long)(n + e20 / 5 % 2) * sR) * 5 + e20 % 5];
#pragma unroll
          for (int i = 0; i < 7; i++) {                // line, row, value
            const int e = min(i * 64 + lane, 403), c = e / 202, r = e % 202 >= 126, k = e % 202 - 126 * r;
            const long row = line_of(c) * nmem + n + r;
            v[i] = *(k < 60 ? fwd + (row * 60 + k) : bwd + (row * 66 + k - 60 + 50 * r));
          }
#pragma unroll
          for (int i = 0; i < 7; i++)
            if (i * 64 + lane < 404) reinterpret_cast<cx<T> *>(sm + TAIL)[i * 64 + lane] = v[i];
          if (lane < 20) *reinterpret_cast<double2 *>(sm + (TAIL + BREC + lane * 16)) = b;
          return;
        }
        cx<T> v[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const int e = min(i * 64 + lane, 149), c = e / 75;
          v[i] = tail[(TW ? bid * 2 + c : line_of(c)) * 150 + (fw ? 0 : 75) + e % 75];
        }
#pragma unroll
        for (int i = 0; i < 3; i++)
          if (i * 64 + lane < 150) reinterpret_cast<cx<T> *>(sm + TAIL)[i * 64 + lane] = v[i];
      };
      // PER, forward: the border sums of a finished chunk.  Lane e of 50 takes
      // entry e of every row's p2 (border row, component, column e % 5) and
      // sums its product with the row's y.  Rows are summed in four classes,
      // (row / G) % 4 with G the shortest chunk of the precision, a class by
      // one wave; classes and columns are added at the end: so all forms of
      // the kernel round alike
      constexpr int G = sizeof(T) == 8 ? 3 : 6;
      static_assert(!PER || R == G || R == 2 * G, "a wave's chunks hold two classes");
      cx<T> bacc[2][2] = {{{0, 0}, {0, 0}}, {{0, 0}, {0, 0}}};      // the wave's classes, the lines
      auto border_sum = [&](int k, int rb) {
        if constexpr (PER) {
          const int e = min(lane, 49), nr = min(R, n - k * R);
          const char *row = sm + (row_off(rb, 0, k * R) + e % 5 * 16);
          const char *row1 = sm + (row_off(rb, 1, k * R) + e % 5 * 16);
          const cx<T> *blk = reinterpret_cast<const cx<T> *>(sm + (BORD + rb * 2 * BORDB)) + e;
          auto add = [&](auto H, int u) {              // row u of both lines, class H of the wave
            cx<T>(&acc)[2] = bacc[decltype(H)::value];
            acc[0] = cfma(blk[u * 50], *reinterpret_cast<const cx<T> *>(row + u * ROWB), acc[0]);
            acc[1] = cfma(blk[u * 50 + R * 50], *reinterpret_cast<const cx<T> *>(row1 + u * ROWB), acc[1]);
          };
          if (R == 2 * G) {
            if (nr == R)
              static_for<R>([&](auto U) { add(idx_t<(decltype(U)::value >= G)>(), decltype(U)::value); });
            else
              for (int u = 0; u < nr; u++) {
                if (u < G) add(idx_t<0>(), u);
                else add(idx_t<1>(), u);
              }
          } else if ((k >> 1) & 1) {
            for (int u = 0; u < nr; u++) add(idx_t<1>(), u);
          } else {
            for (int u = 0; u < nr; u++) add(idx_t<0>(), u);
          }
        }
      };
      // rows n-2 and n-1 of both lines (one wave; lane a of ten has line a / 5
      // and component a % 5): the forward rows with the border sums, then the
      // backward ones, which become the chain's start and the qp terms' x.
      // Every line waits for it, so a loop's LDS reads are in flight together
      // (one at a time they cost a solve 1.4 us: 1025 lines of 24 rows 35.5 ->
      // 32.9 us with the copy of the right-hand side, a step of 257x97 with
      // periodic xi lines 100.5 -> 99.0)
      auto border_rows = [&]() {
        if constexpr (PER) {
          auto *bs = reinterpret_cast<cx<T> *>(sm + TAIL + BSUM);
          const auto *part = reinterpret_cast<const cx<T> *>(sm + TAIL + BPART);
          if (lane < 20) {
            cx<T> t{0, 0};                             // over four classes and five columns
#pragma unroll 5
            for (int k = 0; k < 20; k++) t = t + part[k / 5 * 100 + lane * 5 + k % 5];
            bs[lane] = t;
          }
          wave_sync();
          const int c = min(lane / 5, 1), mm = lane % 5;
          auto *xs = reinterpret_cast<cx<T> *>(sm + SV) + c * 10;      // y_{n-3}, y_{n-4}; then x_{n-2}, x_{n-1}
          const auto *rec = reinterpret_cast<const cx<T> *>(sm + TAIL) + c * 202;
          auto entry = [&](const cx<T> *r, int older, int q) {
            const T *w = reinterpret_cast<const T *>(r) + mm * 20 + rec_pos(older, q);
            return cx<T>{w[0], w[10]};
          };
          auto linv_b = [&](int r) {                   // Linv b, component mm
            const cx<T> *L = rec + r * 126 + 50;
            const double2 *b = reinterpret_cast<const double2 *>(sm + (TAIL + BREC)) + (c * 2 + r) * 5;
            cx<T> acc{(T)b[mm].x, (T)b[mm].y};
#pragma unroll
            for (int q = 0; q < 4; q++) {
              const cx<T> t = cfma(L[min(mm * (mm - 1) / 2 + q, 9)], cx<T>{(T)b[q].x, (T)b[q].y}, acc);
              if (q < mm) acc = t;
            }
            return acc;
          };
          auto uinv = [&](int r, const cx<T> *y) {
            const cx<T> *U = rec + (r ? 186 : 110);
            cx<T> acc{0, 0};
#pragma unroll
            for (int q = 0; q < 5; q++) {
              const cx<T> t = cfma(U[min(mm * 5 - mm * (mm - 1) / 2 + q, 14)], y[min(mm + q, 4)], acc);
              if (q < 5 - mm) acc = t;
            }
            return acc;
          };
          cx<T> y0 = linv_b(0) + bs[c * 10 + mm], y1 = linv_b(1) + bs[c * 10 + 5 + mm];
#pragma unroll 1
          for (int q = 0; q < 5; q++) {
            y0 = cfma(entry(rec, 0, q), xs[q], y0);
            y0 = cfma(entry(rec, 1, q), xs[5 + q], y0);
            y1 = cfma(entry(rec + 126, 1, q), xs[q], y1);
          }
          // y_{n-2}, y_{n-1} take the place of the border sums
          wave_sync();
          if (lane < 10) bs[c * 10 + mm] = y0;
          wave_sync();
#pragma unroll
          for (int q = 0; q < 5; q++) y1 = cfma(entry(rec + 126, 0, q), bs[c * 10 + q], y1);
          if (lane < 10) bs[c * 10 + 5 + mm] = y1;
          wave_sync();
          const cx<T> x1 = uinv(1, bs + c * 10 + 5);
          cx<T> x0 = uinv(0, bs + c * 10);
          if (lane < 10) xs[5 + mm] = x1;
          wave_sync();
#pragma unroll
          for (int q = 0; q < 5; q++) x0 = cfma(entry(rec + 60, 0, q), xs[5 + q], x0);
          if (lane < 10) {
            xs[mm] = x0;
            if (2 * bid + c < L) {
              double2 *at = rhs + (line_of(c) * sL + (long)n * sR) * 5 + mm;
              at[0] = make_double2(x0.re, x0.im);
              at[sR * 5] = make_double2(x1.re, x1.im);
            }
          }
        }
      };
      // c = Linv b or Uinv y in place, component lq of a row per lane (a
      // row's five lanes are in one wave: all have read before any writes)
      auto prep = [&](bool fw, int k, int buf, int rb) {
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; rnd++) {
          int c, u, j;
          if (my_row(fw, k, rnd, c, u, j)) {
            char *row = sm + (row_off(rb, c, first_row(fw, k, c)) + u * ROWB);
            const cx<T> *rp = reinterpret_cast<const cx<T> *>(sm + (buf * BUFB + c * CHB + u * (fw ? 60 : 66) * CS));
            // a row as staged holds complex double; a resident forward
            // result holds the record precision
            auto val = [&](int q) {
              if (RES && !fw) return *reinterpret_cast<const cx<T> *>(row + q * 16);
              const double2 z = *reinterpret_cast<const double2 *>(row + q * 16);
              return cx<T>{(T)z.x, (T)z.y};
            };
            cx<T> acc;
            if (fw) {
              cx<T> l[4], x[4];
              acc = val(lq);
#pragma unroll
              for (int q = 0; q < 4; q++) {
                l[q] = rp[min(50 + lq * (lq - 1) / 2 + q, 59)];
                x[q] = val(q);
              }
#pragma unroll
              for (int q = 0; q < 4; q++) {
                const cx<T> t = cfma(l[q], x[q], acc);
                if (q < lq) acc = t;
              }
            } else {
              cx<T> v[5], x[5];
              acc = cx<T>{0, 0};
#pragma unroll
              for (int q = 0; q < 5; q++) {
                v[q] = rp[min(50 + lq * 5 - lq * (lq - 1) / 2 + q, 64)];
                x[q] = val(min(lq + q, 4));
              }
#pragma unroll
              for (int q = 0; q < 5; q++) {
                const cx<T> t = cfma(v[q], x[q], acc);
                if (q < 5 - lq) acc = t;
              }
              if constexpr (PER) {                     // what x_{n-2}, x_{n-1} add
                const cx<T> *xb = reinterpret_cast<const cx<T> *>(sm + SV) + c * 10;
                const cx<T> *blk = reinterpret_cast<const cx<T> *>(sm + (BORD + (rb * 2 + c) * BORDB)) + u * 50 + lq * 5;
                cx<T> e{0, 0};
#pragma unroll
                for (int q = 0; q < 5; q++) {
                  acc = cfma(blk[q], xb[q], acc);
                  e = cfma(blk[25 + q], xb[5 + q], e);
                }
                acc = acc + e;
              }
            }
            *reinterpret_cast<cx<T> *>(row + lq * 16) = acc;
          }
        }
      };
      // the results of a chunk to memory
      auto copy_out = [&](bool fw, int k, int rb) {
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; rnd++) {
          int c, u, j;
          if (my_row(fw, k, rnd, c, u, j) && (TW || 2 * bid + c < L)) {
            const cx<T> x =
                *reinterpret_cast<const cx<T> *>(sm + (row_off(rb, c, first_row(fw, k, c)) + u * ROWB + lq * 16));
            *value_of(rhs, c, j) = make_double2(x.re, x.im);
            if (PER && !fw && j == 0) rhs[(line_of(c) * sL + (long)nmem * sR) * 5 + lq] = make_double2(x.re, x.im);
          }
        }
      };
      // Wave 1 starts the copies: a chunk's NBUF - 1 iterations before it is
      // computed, when its buffer's last chunk is done, and waits two
      // iterations before, so that chunks are in flight for NBUF - 2
      // iterations.  Waves 2 and 3 take turns to prepare the chunk one ahead
      // of the compute wave and to copy out the chunk two behind it (the
      // compute wave's barriers don't wait for its last write).
      constexpr int OPS = 2 * ((R * 60 * (int)CS + 1023) / 1024 + (PER ? (R * 50 * (int)CS + 1023) / 1024 : 0)) + (RES ? 0 : ROUNDS);   // copies of a full chunk, at least
      constexpr int AHEAD = (NBUF - 3) * OPS < 63 ? (NBUF - 3) * OPS : 63;   // copies younger than those waited for (a six-bit counter)
      // both passes are one stream of chunks where the right-hand sides are
      // resident (the backward pass's first chunk is prepared between them);
      // else one stream each, as the backward pass reads what the forward
      // pass wrote
      const int M = RES ? 2 * N : N;
#pragma unroll 1
      for (int pass = 0; pass < (RES ? 1 : 2); pass++) {
        auto is_fw = [&](int c) { return RES ? c < N : pass == 0; };
        auto kk = [&](int c) { return RES && c >= N ? c - N : c; };
        if (w == 0) {
          // chunks [lo, hi) of a pass are full in both chains
          const int ff = len1 / R, b0 = TW ? 1 : 0, bf = (min(jtop(0), jtop(1)) + 1) / R;
          int lo = RES || pass == 0 ? 0 : b0, hi = RES || pass == 0 ? ff : bf;
          auto wait_for = [&](int K) {                  // chunk K + 2; younger: K + 3 .. K + NBUF - 1
            if (RES && K + 3 == N) {
              lo = N + b0;
              hi = N + bf;
            }
            if (K + 3 >= lo && K + NBUF - 1 < hi) __builtin_amdgcn_s_waitcnt(0x0F70 | (AHEAD & 15) | ((AHEAD >> 4) << 14));
            else __builtin_amdgcn_s_waitcnt(0x0F70);    // vmcnt(0)
          };
          for (int c = 0; c < NBUF - 1 && c < M; c++) issue(is_fw(c), kk(c), c, c);
          wait_for(-1);
          loader_barrier();
          loader_barrier();
          int buf = NBUF - 1, rb = NBUF - 1;
          for (int K = 0; K < M; K++) {
            if (RES && K == N) {
              if (PER) {
                loader_barrier();
                loader_barrier();
              }
              loader_barrier();
            }
            if (K + NBUF - 1 < M) issue(is_fw(K + NBUF - 1), kk(K + NBUF - 1), buf, rb);
            wait_for(K);
            buf = buf + 1 == NBUF ? 0 : buf + 1;
            rb = rb + 1 == NROW ? 0 : rb + 1;
            loader_barrier();
          }
          if (PER && !RES && pass == 0) {
            loader_barrier();
            loader_barrier();
          }
        } else {
          // wave p prepares, sums and writes out the chunks of its parity
          const int p = w - 1;
          // PER: the border between the passes; the last two chunks' sums are
          // still to be added
          auto border = [&]() {
            const int last = ((N - 1) & 1) == p ? N - 1 : N - 2;
            if (last >= 0) border_sum(last, last % NROW);
            if (lane < 50)
              for (int h = 0; h < 2; h++)
                for (int c = 0; c < 2; c++)
                  reinterpret_cast<cx<T> *>(sm + TAIL + BPART)[(R == G ? p + 2 * h : 2 * p + h) * 100 + c * 50 + lane] =
                      bacc[h][c];
            loader_barrier();
            if (p == 0) border_rows();
            loader_barrier();
          };
          if (RES) load_rhs(p, 2);
          if (p == 1 && (!PER || pass == 0)) load_tail(is_fw(0));
          __builtin_amdgcn_s_waitcnt(0);
          loader_barrier();
          if (p == 0) prep(is_fw(0), 0, 0, 0);
          loader_barrier();
          int buf = 1, rb = 1, ro = 0;                  // buffers of chunks K + 1, staging of K - 2
          for (int K = 0; K < M; K++) {
            if (RES && K == N) {
              if (PER) border();
              if (p == 0) prep(false, 0, N % NBUF, N % NROW);
              else load_tail(false);
              loader_barrier();
            }
            if (((K + 1) & 1) == p) {
              if (K + 1 < M && !(RES && K + 1 == N)) prep(is_fw(K + 1), kk(K + 1), buf, rb);
            } else if (K >= 2) {
              if (PER && is_fw(K - 2) && !(RES && K >= N)) border_sum(kk(K - 2), ro);
              if (!RES || K - 2 >= N) copy_out(is_fw(K - 2), kk(K - 2), ro);
            }
            buf = buf + 1 == NBUF ? 0 : buf + 1;
            rb = rb + 1 == NROW ? 0 : rb + 1;
            if (K >= 2) ro = ro + 1 == NROW ? 0 : ro + 1;
            loader_barrier();
          }
          if (N - 2 + p >= 0) copy_out(is_fw(M - 1), N - 2 + p, (N - 2 + p) % NROW);
          if (PER && !RES && pass == 0) border();
          __builtin_amdgcn_s_waitcnt(0);                // a forward pass's results are in memory
        }
        if (!RES) loader_barrier();
      }
      // nothing is in flight here; said again because the compiler carries the
      // copies' pending state into the compute wave's code otherwise, where it
      // then waits for every LDS read before each step
      __builtin_amdgcn_s_waitcnt(0);
      return;
    }

    // ---- compute wave ----
    // Its priority is raised: where it shares a SIMD with loader waves of
    // another workgroup they would take issue slots from it.
    // 16-lane row r: chain r & 1, half r >> 1.  Lanes 0-4 of a row hold the
    // real parts of the components, lanes 5-9 the imaginary ones (the lanes
    // past 9 repeat lane 9).  The lower half sums c + W2 y_{i-1}, the upper
    // half W1 y_{i-2}; V holds y_{i-1} below and y_{i-2} above.
    __builtin_amdgcn_s_setprio(3);
    const int ch = (lane >> 4) & 1, hq = lane >> 5, l9 = min(lane & 15, 9), im = l9 >= 5, m = l9 - 5 * im;
    const T low = hq ? T(0) : T(1), sgn = im ? T(1) : T(-1);
    constexpr unsigned ES = sizeof(T);
    for (int e = lane; e < R * 5; e += 64) *reinterpret_cast<double2 *>(sm + (ZERO + e * 16)) = make_double2(0.0, 0.0);
    T V = 0;
    T ar[3][5], br[3][5], cr[3];
    // a lane's offsets in a record row (rec_pos): pairs and last column of
    // the parts that meet real and imaginary broadcasts
    const unsigned wa = ch * CHB + (20 * m + 10 * im + 2 * hq) * ES, wb = ch * CHB + (20 * m + 10 * (1 - im) + 2 * hq) * ES;
    const unsigned last = 8 * ES - hq * ES;
    typedef T pair_t __attribute__((ext_vector_type(2)));
    auto ld5 = [&](unsigned at, unsigned at4, unsigned row, T (&x)[5]) {
      const pair_t p = *reinterpret_cast<const pair_t *>(sm + (at + row));
      const pair_t q = *reinterpret_cast<const pair_t *>(sm + (at + row + 4 * ES));
      x[0] = p.x;
      x[1] = p.y;
      x[2] = q.x;
      x[3] = q.y;
      x[4] = *reinterpret_cast<const T *>(sm + (at4 + row));
    };
    auto sv = [&](int c, int k) { return reinterpret_cast<cx<T> *>(sm + SV) + (c * 2 + k) * 5; };
    auto sv_lane = [&](int c, int k) -> T & { return *reinterpret_cast<T *>(sm + (SV + ((c * 2 + k) * 5 + m) * CS + im * ES)); };
    const cx<T> *tl = reinterpret_cast<const cx<T> *>(sm + TAIL) + ch * 75 + m * 5;

    auto pass = [&](auto FWT, int K0) {
      constexpr bool FW = decltype(FWT)::value;
      constexpr unsigned ROW = (FW ? 60 : 66) * CS;
      V = PER && !FW ? sv_lane(ch, hq) : T(0);      // PER: the backward chain starts from x_{n-2}, x_{n-1}
      const int jt = jtop(ch);
      // chunks of ordinary steps only: both chains active, no hand-off, no
      // boundary block, no value to keep
      const int main_lo = (!FW && TW) ? 1 : 0;
      const int main_hi = PER ? n : FW ? (TW ? len1 : n - 3) : min(jtop(0), jtop(1)) - 2;
      // LDS offsets of a chunk for this lane: records (real, imaginary
      // broadcasts; their last columns), c read, result written
      struct At { unsigned a, a4, b, b4, c, y; };
      auto at_chunk = [&](int k, int buf, int rb) {
        const unsigned r = row_off(rb, ch, FW ? k * R : jt - k * R - R + 1), d = buf * BUFB;
        const unsigned e = m * 16 + im * ES;
        return At{d + wa, d + wa + last, d + wb, d + wb + last, (hq ? ZERO : r) + e, (hq ? DUMMY : r) + e};
      };
      auto load = [&](const At &t, int slot, T (&a)[5], T (&b)[5]) {
        ld5(t.a, t.a4, slot * ROW, a);
        ld5(t.b, t.b4, slot * ROW, b);
      };
      auto load_c = [&](const At &t, int slot) { return *reinterpret_cast<const T *>(sm + (t.c + slot * ROWB)); };
      // one step: c is added last in every form of the kernel, so that all
      // round alike
      auto step = [&](const At &t, int slot, const T (&a)[5], const T (&b)[5], T c) {
        T x = 0, y = 0;
        row_mac5(x, y, V, a, b);
        V = hand_over(T(fma(y, sgn, x + c)), V, low);
        *reinterpret_cast<T *>(sm + (t.y + slot * ROWB)) = V;
      };
      // main chunks [k0, k1)
      const int k0 = min(main_lo, N), k1 = max(k0, main_hi / R);
      int buf = K0 % NBUF, rb = 0;
      auto next_chunk = [&](bool wait) {
        buf = buf + 1 == NBUF ? 0 : buf + 1;
        rb = rb + 1 == NROW ? 0 : rb + 1;
        if (wait) {
          loader_barrier();
        } else {                 // the last write is read two iterations on
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        }
      };
      auto plain = [&](int k) {
        const At now = at_chunk(k, buf, rb);
        const int s_end = min(k * R + R, len0);
        for (int s = k * R; s < s_end; s++) {
          const int slot = FW ? s - k * R : R - 1 - (s - k * R);
          const int j = FW ? s : jt - s;
          if (FW && TW && s == len1) {               // chain 1 is done: its last rows h+2, h+3
            if (ch == 1) sv_lane(0, hq) = V;
            wave_sync();
          }
          if (FW && !TW && !PER && s == n - 3) {     // rows n-5, n-4
            sv_lane(ch, 1 - hq) = V;
            wave_sync();
          }
          if (!FW && TW && s == 2) {                 // chain 1 starts from x_h, x_{h+1}
            if (ch == 0) sv_lane(1, hq) = V;
            wave_sync();
            if (ch == 1) V = sv_lane(1, 1 - hq);
            wave_sync();
          }
          if (!FW && !PER && j == 2) sv_lane(ch, hq) = V;    // chain rows 3, 4
          if (!FW) wave_sync();
          T a[5], b[5];
          load(now, slot, a, b);
          T c = load_c(now, slot);
          // blocks of the pass's last two rows outside the band
          const bool ends = PER ? false : FW ? (s >= len0 - 2 && (!TW || ch == 0)) : (j == 0 || j == 1);
          if (ends && hq == 0) {
            const int from = FW && TW ? 0 : ch;
            const bool end = FW ? s == len0 - 1 : j == 0;
            const cx<T> *t1 = tl + (end ? 25 : FW ? 0 : 50), *x1 = sv(from, FW ? 0 : 1);
            cx<T> e{0, 0};
#pragma unroll
            for (int q = 0; q < 5; q++) e = cfma(t1[q], x1[q], e);
            if (end) {
              const cx<T> *t2 = tl + (FW ? 50 : 0), *x2 = sv(from, FW ? 1 : 0);
#pragma unroll
              for (int q = 0; q < 5; q++) e = cfma(t2[q], x2[q], e);
            }
            c += im ? e.im : e.re;
          }
          step(now, slot, a, b, c);
        }
        next_chunk(k + 1 == N);
      };
      for (int k = 0; k < k0; k++) plain(k);
      if (k1 > k0) {
        At now = at_chunk(k0, buf, rb);
        load(now, FW ? 0 : R - 1, ar[0], br[0]);
        load(now, FW ? 1 : R - 2, ar[1], br[1]);
        for (int k = k0; k < k1; k++) {
          // the first two rows' records, read in the last iteration, are here
          // (all but the last write done)
          __builtin_amdgcn_s_waitcnt(0xC17F);
          now = at_chunk(k, buf, rb);
          // records two steps ahead of use, in three rotating register sets;
          // past the last chunk they are read and not used.  c of the chunk's
          // first rows was formed in the last iteration and is read now
          const At next = at_chunk(k + 1, buf + 1 == NBUF ? 0 : buf + 1, 0);
          cr[0] = load_c(now, FW ? 0 : R - 1);
          cr[1] = load_c(now, FW ? 1 : R - 2);
          static_for<R>([&](auto U) {
            constexpr int u = decltype(U)::value, s0 = u % 3, s2 = (u + 2) % 3;
            constexpr int u2 = (u + 2) % R, slot2 = FW ? u2 : R - 1 - u2;
            if constexpr (u + 2 < R) {
              load(now, slot2, ar[s2], br[s2]);
              cr[s2] = load_c(now, slot2);
            } else {
              load(next, slot2, ar[s2], br[s2]);
            }
            step(now, FW ? u : R - 1 - u, ar[s0], br[s0], cr[s0]);
          });
          next_chunk(k + 1 == N);
        }
      }
      for (int k = k1; k < N; k++) plain(k);
    };
    loader_barrier();
    loader_barrier();
    pass(std::true_type{}, 0);
    if (PER) {
      sv_lane(ch, hq) = V;    // y_{n-3}, y_{n-4}, for the rows the loader waves solve now
      loader_barrier();
      loader_barrier();
    }
    loader_barrier();         // RES: the backward pass's first chunk is prepared; else the results are in memory
    if (!RES) {
      loader_barrier();
      loader_barrier();
    }
    pass(std::false_type{}, RES ? N : 0);
    if (!RES) loader_barrier();
  }
};

// the lines of one plan; neighbouring lines, which share cache lines of the
// right-hand side where rows are far apart, on one XCD
template <typename T, int R, int NBUF, bool TW, bool RES>
__global__ __launch_bounds__(256, 2) void k_line_solve(int n, int h, long L, const cx<T> *__restrict__ fwd,
                                                      const cx<T> *__restrict__ bwd, const cx<T> *__restrict__ tail,
                                                      const double2 *in, double2 *rhs, long sL, long sR) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  LineSolve<T, R, NBUF, TW, RES>::run(sm, xcd_tile(blockIdx.x, gridDim.x), n, h, L, fwd, bwd, tail, in, rhs, sL, sR);
}

// periodic lines
template <typename T, int R, int NBUF, bool RES>
__global__ __launch_bounds__(256, 2) void k_line_solve_per(int n, long L, const cx<T> *__restrict__ fwd,
                                                          const cx<T> *__restrict__ bwd, const cx<T> *__restrict__ p2,
                                                          const cx<T> *__restrict__ qp, const double2 *in,
                                                          double2 *rhs, long sL, long sR) {
  extern __shared__ __attribute__((aligned(16))) char sm[];
  LineSolve<T, R, NBUF, false, RES, true>::run(sm, xcd_tile(blockIdx.x, gridDim.x), n, -1, L, fwd, bwd, nullptr, in, rhs,
                                               sL, sR, p2, qp);
}

}  // namespace lns3d
