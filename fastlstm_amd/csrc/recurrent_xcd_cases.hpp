// The instances of the XCD-local kernels: one list for what is compiled (recurrent_xcd_inst.inc) and for what a shape may be given
// (xcd_shape in api.hip).
#pragma once

namespace fastlstm {

// lstm_fwd_xcd_kernel<T, MT, NKW, NTW, NWV>.  fp32: three parts of every weight; 32 units per workgroup (MT = 8) up to H = 256, where
// the batch has more tiles than groups of 16 units (H = 256: from 513 rows on).
#define FASTLSTM_FWD_XCD_16(X) \
    X(2, 4, 1, 4) X(2, 4, 2, 4) X(2, 8, 1, 4) X(2, 8, 2, 4) X(4, 4, 1, 4) X(4, 4, 2, 4) X(4, 8, 1, 4) X(4, 8, 2, 4) \
    X(8, 4, 1, 4) X(8, 4, 2, 4) X(8, 8, 1, 8) X(8, 8, 2, 8)
#define FASTLSTM_FWD_XCD_32(X) \
    X(2, 2, 1, 4) X(2, 2, 2, 4) X(4, 2, 1, 4) X(4, 2, 2, 4) X(8, 2, 1, 8) X(8, 2, 2, 8) X(4, 4, 1, 8) X(4, 4, 2, 8)
// lstm_bwd_xcd_kernel<T, MT, NKW, NTW, 8>
#define FASTLSTM_BWD_XCD_16(X) \
    X(1, 4, 1) X(1, 4, 2) X(1, 8, 1) X(1, 8, 2) X(1, 16, 1) X(1, 16, 2) X(2, 4, 1) X(2, 4, 2) X(2, 8, 1) X(2, 8, 2) X(2, 16, 1) X(2, 16, 2)
#define FASTLSTM_BWD_XCD_32(X) \
    X(1, 2, 1) X(1, 2, 2) X(1, 4, 1) X(1, 4, 2) X(1, 8, 1) X(1, 8, 2) X(2, 2, 1) X(2, 2, 2) X(2, 4, 1) X(2, 4, 2)

constexpr bool xcd_instance_exists(bool fp32, bool backward, int mt, int nkw, int ntw, int nwv) {
#define X4(MT, NKW, NTW, NWV) if (mt == MT && nkw == NKW && ntw == NTW && nwv == NWV) return true;
#define X3(MT, NKW, NTW) if (mt == MT && nkw == NKW && ntw == NTW && nwv == 8) return true;
    if (backward) {
        if (fp32) { FASTLSTM_BWD_XCD_32(X3) } else { FASTLSTM_BWD_XCD_16(X3) }
    } else {
        if (fp32) { FASTLSTM_FWD_XCD_32(X4) } else { FASTLSTM_FWD_XCD_16(X4) }
    }
#undef X3
#undef X4
    return false;
}

}  // namespace fastlstm
