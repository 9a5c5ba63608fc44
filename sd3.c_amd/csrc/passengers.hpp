// How many modulation panels (common.hpp: AdaWork) the workgroups that a launch adds on its idle compute units may take along. Host code only.
#pragma once

namespace sd3 {

// us until such a workgroup has started and has the rows of y in LDS
constexpr double PASSENGER_START = 6.0;
// us that a panel of K x 64 weights from HBM takes it. A slice of K is K / 32 rows, requested 16 at a time, so what counts is the groups of 512 k
// values. Alone on a device, 64 workgroups of 512 threads, one row of y, K = 512, 768, 1024, 1536, 2048, 2432, 3072, 4096: 2.4, 4.0, 4.0, 5.7, 7.3, 9.0, 10.3,
// 12.9 (two and four rows within 8 % of that, 160 workgroups 0.1 to 0.6 more, from 2048 on 1 to 3.5); beside the launch's own workgroups at
// K = 1536 about 6.5, and the others in proportion. With 6.5 for every K launches of width 768 left a third of their room and those of 2432 and 3072 were
// outlasted by their passengers. Forwards, us, 6.5 | so | without passengers: width 768, 512px 2319 | 2283 | 2368; width 2432, eight blocks, 256px 1570 | 1538 |
// 1667, batch 4 2997 | 2732 | 3058, 512px 2903 | 2724 | 3040; width 3072, six blocks, 256px 1689 | 1628 | 1878, 512px 3158 | 2855 | 3033, batch 2
// 4573 | 4353 | 4499.
inline double passenger_panel_us(int K) { return 1.0 + 11.0 / 6.0 * ((K + 511) / 512); }
// A block's last launch may take up to this much more: what is left of the panels would be a launch of its own (512px at width 1536: 2.8 % of a forward),
// and the cost table is a quarter below what a launch with 96 K tiles takes beside the others.
constexpr double PASSENGER_OVERTIME = 32.5;

// Panels for each of `idle` workgroups of a launch that takes `us`, of `want` panels in all: as many as it has time for
inline int passenger_panels(double us, int K, int want, int idle, bool last) {
    if (want <= 0 || idle <= 0) return 0;
    const double panel = passenger_panel_us(K), time = us - PASSENGER_START;
    const int rest = (want + idle - 1) / idle;
    if (last && rest * panel <= time + PASSENGER_OVERTIME) return rest;
    const int room = time > 0 ? (int)(time / panel) : 0;
    return room < rest ? room : rest;
}

// Whether taking panels along is worth a launch for those that nobody had room for: it costs about 6 us beside its streaming, the launch up front that
// does them all streams 5.4 TB/s. A forward whose blocks take fewer along than that does all the others in one launch instead. Width 768, 256px, batch 4
// (launches of 252 tiles on 256 units, 144 or 180 panels of 98 KB a block): 2203 us with all of them up front, 2310 with a launch per block, 2186 so.
inline bool passengers_pay(int taken, int K) { return taken * (K * 128.0 / 5.4e6) >= 6.0; }

}  // namespace sd3
