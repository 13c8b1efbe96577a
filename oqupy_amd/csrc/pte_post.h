// Posts of the pivoted QR (qrcp_kernel): what a workgroup tells the others of a
// step, in words that each carry the step's tag.
#pragma once

// Bits of two non-negative doubles, which order as the values do.
struct QrcpPost {
  unsigned long long norm;   // largest residual norm of the workgroup's columns
  unsigned long long sum;    // sum of their squared residual norms
  unsigned local;            // the norm's column among the workgroup's own, < kQrNoColumn
};                           // (that: none is left)

// Words 0 and 1, which everyone reads every step, hold the sum, the upper half of
// the norm and the column; word 2 the lower half of the norm, which decides, and is
// read, only where upper halves tie. (996 x 860, 215 workgroups: 9.0 us a step;
// with three words read every step 9.3, and 10.0 with word k of all workgroups
// together, where many workgroups write one line that all are reading.)
constexpr int kQrPostWords = 3;
constexpr unsigned kQrNoColumn = 0xffu;
constexpr unsigned long long kQrTagMask = 0xfffull;

// tag of step j: never 0, and not that of step j - 2, which has the same place
constexpr unsigned long long qrcp_tag(int j) { return (unsigned long long)(1 + j % 4095); }

constexpr bool qrcp_tagged(unsigned long long word, unsigned long long tag) {
  return (word & kQrTagMask) == tag;
}

constexpr unsigned long long qrcp_word(const QrcpPost& p, int k, unsigned long long tag) {
  return (k == 0   ? p.sum & ~kQrTagMask
          : k == 1 ? (p.norm >> 32) << 32 | (unsigned long long)p.local << 24 |
                         (p.sum & kQrTagMask) << 12
                   : p.norm << 32) |
         tag;
}

// without the lower half of the norm
constexpr QrcpPost qrcp_unpack(unsigned long long w0, unsigned long long w1) {
  return QrcpPost{(w1 >> 32) << 32, (w0 & ~kQrTagMask) | ((w1 >> 12) & kQrTagMask),
                  (unsigned)(w1 >> 24) & kQrNoColumn};
}
constexpr unsigned qrcp_norm_low(unsigned long long w2) { return (unsigned)(w2 >> 32); }
