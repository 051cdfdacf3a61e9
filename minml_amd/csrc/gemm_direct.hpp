/*
 * gemm_direct.hpp — fp16 products too small to give every compute unit a streaming workgroup:  C[i] = A[i] * B[i]^T  with short K rows
 * (the 36 Winograd products of a few positions; the dense layers and 1x1 convolutions of a few positions).
 *
 * Such a launch is bound by latency, not by HBM or the matrix cores: it takes one memory round trip, the bytes that the busiest compute
 * unit must pull in, a short chain of MFMAs and the stores. The streaming kernel (gemm_stream.hpp) is the wrong shape for it: a
 * workgroup there first brings 128 KB of B into registers, 32 rows x 32 bytes per instruction, and at one position all but 36 compute
 * units stay idle. Here the product is cut into tiles small enough to occupy the chip, and a workgroup requests the WHOLE K extent of
 * its rows of A and B at once by direct-to-LDS loads (8 rows x 128 bytes per instruction, whole cache lines; the same loads straight
 * into the fragment layout, 16 half lines per instruction, took 13.9 instead of 7.1 us at 256 rows), multiplies each 128-byte piece of
 * K as soon as it has landed (one barrier per piece), and stores its 4 consecutive outputs per lane and block directly.
 * 16x16 MFMA blocks (v_mfma_f32_16x16x32_f16: bit-identical to the 32x32x16 form of the other engines, so that a position's result does
 * not depend on which engine its batch takes). Two tile shapes: 64 x 64 by 8 wavefronts of 16 x 32 (many small wavefronts keep more
 * loads in flight: 4 wavefronts of 32 x 32 take 7.05 instead of 6.66 us at 256 rows), and 32 x 32 by 4 wavefronts of 16 x 16 where
 * 64 x 64 leaves compute units without a tile. Consecutive tiles (same matrix, same columns) lie on one XCD and share its L2.
 *
 * The first loads wait for the workgroup's tile: its numbers come from divisors prepared on the host (TileOrder), rows of A and B are different loads, so that no
 * lane chooses between them, and everything else is asked for with one set of scalar loads. 344 -> 193 instructions, 162 -> 90 of them before the first load;
 * from a workgroup's start until its loads are out 0.9 -> 0.5 us, the launch 2.6 -> 2.2 us (timestamps in the kernel, one 15x15 position of 256 channels).
 *
 * Measured, 36 products of M rows, 8 launches replayed as one graph, us per launch, streaming kernel (384-byte rows: tile engine) ->
 * this one: 64 -> 64 channels: M = 16 (one 15x15 position) 4.6 -> 3.4, 1024 6.0 -> 5.5; 128 -> 128: 16 6.0 -> 3.4, 512 7.2 -> 5.7;
 * 192 -> 192: 16 4.4 -> 3.5, 256 6.5 -> 5.1, 1024 20.0 -> 11.1, 2048 39.2 -> 20.5, 16384 202 -> 163; 256 -> 256: 16 9.8 -> 4.0,
 * 64 10.0 -> 4.2, 256 9.7 -> 6.8, 512 14.0 -> 9.9; 384 -> 384: 16 11.4 -> 4.1, 128 12.3 -> 7.7, 256 13.7 -> 12.1. One product of 256 -> 768
 * columns: 225 rows 9.7 -> 2.9, 1350 10.2 -> 4.7, 4000 10.1 -> 8.5.
 */
#ifndef MINML_AMD_GEMM_DIRECT_HPP_
#define MINML_AMD_GEMM_DIRECT_HPP_

#include "common.hpp"
#include "gemm_stream.hpp"
#include "gemm_tiles.hpp"

namespace mlhip
{
	template<int KB, int BLOCKS_M, int BLOCKS_N, int WAVES_M, int WAVES_N, typename Epilogue>
	__global__ __launch_bounds__(64 * WAVES_M * WAVES_N) void kernel_gemm_direct_nt(const half_t *A, const half_t *B, half_t *C, int M, int N, size_t stride_a,
			size_t stride_b, size_t stride_c, TileOrder order, uint32_t a_row_bytes, Epilogue epilogue)
	{
		constexpr bool PLAIN = std::is_same<Epilogue, PlainStore>::value;
		constexpr int PIECES = KB / 128; /* 128-byte pieces of a K row */
		constexpr int BM = 16 * BLOCKS_M * WAVES_M, BN = 16 * BLOCKS_N * WAVES_N, WAVES = WAVES_M * WAVES_N;
		constexpr int ROW_BLOCKS = (BM + BN) / 8; /* 8-row blocks of a piece */
		constexpr int A_LOADS = BM / 8 / WAVES, B_LOADS = BN / 8 / WAVES, PIECE_LOADS = A_LOADS + B_LOADS; /* of them per wavefront */
		static_assert(KB % 128 == 0 && BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "K rows of whole 128-byte pieces, the same loads for every wavefront");
		static_assert(WAVES % 2 == 0, "the swizzle of a lane is then the same in all its loads");
		const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
		const int wave_m = wave / WAVES_N, wave_n = wave % WAVES_N;
		const int frag_row = lane & 15, quarter = lane >> 4;

		const TileOrder::Tile tile = order.tile_of(blockIdx.x);
		const unsigned int matrix = tile.matrix;
		const int m_tile = tile.row * BM, n_tile = tile.column * BN;
		const int m0 = m_tile + wave_m * 16 * BLOCKS_M, n0 = n_tile + wave_n * 16 * BLOCKS_N;

		/* lane l, register r of block (i, j): m = 16 i + l % 16, n = 16 j + 4 (l / 16) + r */
		Epilogue local = epilogue;
		struct Nothing
		{
				struct Column
				{
				};
				struct Extra
				{
				};
		};
		typedef typename std::conditional<PLAIN, Nothing, Epilogue>::type Parts;
		typename Parts::Column column[BLOCKS_N];
		typename Parts::Extra extra[BLOCKS_M][BLOCKS_N];
		if constexpr (!PLAIN)
		{
			local.D += matrix * stride_c;
			if (local.bias != nullptr)
				local.bias += static_cast<size_t>(matrix) * local.bias_batch_stride;
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
			{
				const int n = n0 + 16 * j + 4 * quarter;
				column[j] = local.load_column(n < N ? n : 0);
			}
			if (local.has_extra())
			{
				local.C += matrix * stride_c;
#pragma unroll
				for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
					for (int j = 0; j < BLOCKS_N; j++)
					{
						const int n = n0 + 16 * j + 4 * quarter;
						extra[i][j] = local.load_extra(min(m0 + 16 * i + frag_row, M - 1), n < N ? n : 0);
					}
			}
		}

		/* operand tiles -> LDS: [128-byte piece of K][row][128 bytes], 8 rows per instruction, the 16-byte chunks of a row swizzled */
		extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
		const uint8_t *a_base = reinterpret_cast<const uint8_t*>(A + matrix * stride_a);
		const uint8_t *b_base = reinterpret_cast<const uint8_t*>(B + matrix * stride_b);
		const int sub_row = lane >> 3, chunk = ((lane & 7) ^ ((4 * wave + (sub_row >> 1)) & 7)) * 16;
		const uint8_t *src[PIECE_LOADS];
#pragma unroll
		for (int u = 0; u < A_LOADS; u++)
			src[u] = a_base + static_cast<uint64_t>(static_cast<uint32_t>(min(m_tile + (wave + WAVES * u) * 8 + sub_row, M - 1))) * a_row_bytes + chunk;
#pragma unroll
		for (int u = 0; u < B_LOADS; u++)
			src[A_LOADS + u] = b_base + static_cast<uint64_t>(static_cast<uint32_t>(min(n_tile + (wave + WAVES * u) * 8 + sub_row, N - 1))) * KB + chunk;
#pragma unroll
		for (int piece = 0; piece < PIECES; piece++)
#pragma unroll
			for (int u = 0; u < PIECE_LOADS; u++)
				__builtin_amdgcn_global_load_lds((global_ptr_t) (src[u] + piece * 128), (lds_ptr_t) (lds + (piece * ROW_BLOCKS + wave + WAVES * u) * 1024), 16, 0, 0);
		float4_t acc[BLOCKS_M][BLOCKS_N];
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
				acc[i][j] = float4_t { 0.0f, 0.0f, 0.0f, 0.0f };
		int a_first[BLOCKS_M], b_first[BLOCKS_N]; /* this lane's fragment of the first k step, the others by XOR and piece */
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
		{
			const int row = wave_m * 16 * BLOCKS_M + 16 * i + frag_row;
			a_first[i] = row * 128 + ((quarter ^ ((row >> 1) & 7)) * 16);
		}
#pragma unroll
		for (int j = 0; j < BLOCKS_N; j++)
		{
			const int row = BM + wave_n * 16 * BLOCKS_N + 16 * j + frag_row;
			b_first[j] = row * 128 + ((quarter ^ ((row >> 1) & 7)) * 16);
		}
		stream_static_for<2 * PIECES>([&](auto step)
		{
			constexpr int s = decltype(step)::value;
			if constexpr (s % 2 == 0)
			{ /* piece s / 2 has landed once at most the loads of the later pieces are outstanding (loads return in order) */
				wait_vmcnt<(PIECES - 1 - s / 2) * PIECE_LOADS>();
				barrier_no_fence();
			}
			uint4_t a[BLOCKS_M], b[BLOCKS_N];
			const uint8_t *piece = lds + (s / 2) * (BM + BN) * 128;
#pragma unroll
			for (int i = 0; i < BLOCKS_M; i++)
				a[i] = *reinterpret_cast<const uint4_t*>(piece + (a_first[i] ^ ((s & 1) * 64)));
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
				b[j] = *reinterpret_cast<const uint4_t*>(piece + (b_first[j] ^ ((s & 1) * 64)));
#pragma unroll
			for (int i = 0; i < BLOCKS_M; i++)
#pragma unroll
				for (int j = 0; j < BLOCKS_N; j++)
					acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, b[j]), __builtin_bit_cast(half8_t, a[i]), acc[i][j], 0, 0, 0);
		});
#pragma unroll
		for (int i = 0; i < BLOCKS_M; i++)
		{
			const int m = m0 + 16 * i + frag_row;
			if (m >= M)
				continue;
#pragma unroll
			for (int j = 0; j < BLOCKS_N; j++)
			{
				const int n = n0 + 16 * j + 4 * quarter;
				if (n >= N) /* N is a multiple of 4 (checked by the launcher) */
					continue;
				if constexpr (PLAIN)
				{
					Vec<half_t, 4> out;
#pragma unroll
					for (int e = 0; e < 4; e++)
						out.v[e] = acc[i][j][e];
					out.store(C + matrix * stride_c + static_cast<size_t>(m) * N + n);
				}
				else
				{
					const float vals[4] = { acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3] };
					local.apply(m, n, vals, column[j], extra[i][j]);
				}
			}
		}
	}

	template<int KB, int BLOCKS_M, int BLOCKS_N, int WAVES_M, int WAVES_N, typename Epilogue>
	inline void launch_gemm_direct_as(hipStream_t stream, const StreamGemmArgs &g, const Epilogue &epilogue)
	{
		const int tiles_m = ceil_div(g.M, 16 * BLOCKS_M * WAVES_M), tiles_n = ceil_div(g.N, 16 * BLOCKS_N * WAVES_N);
		constexpr int LDS = KB * 16 * (BLOCKS_M * WAVES_M + BLOCKS_N * WAVES_N);
		auto kernel = kernel_gemm_direct_nt<KB, BLOCKS_M, BLOCKS_N, WAVES_M, WAVES_N, Epilogue>;
		if (LDS > 64 * 1024)
			ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), LDS);
		const TileOrder order = make_tile_order(products_meet_in_l2(g, sizeof(half_t)) ? TileOrder::MATRICES_BETWEEN : TileOrder::ROWS_INNERMOST, tiles_m, tiles_n, g.batch);
		hipLaunchKernelGGL(kernel, dim3(order.tiles), dim3(64 * WAVES_M * WAVES_N), LDS, stream, reinterpret_cast<const half_t*>(g.A),
				reinterpret_cast<const half_t*>(g.B), reinterpret_cast<half_t*>(g.C), g.M, g.N, g.stride_a, g.stride_b, g.stride_c, order,
				g.a_row_bytes != 0 ? static_cast<uint32_t>(g.a_row_bytes) : static_cast<uint32_t>(KB), epilogue);
	}
	/*
	 * Whether this kernel takes a product: the 64 x 64 tiles per compute unit up to which it is not behind the kernel that would take it
	 * otherwise. Every tile fetches its rows of A and B anew (KB * 128 bytes) where the streaming kernel fetches A once. Single products
	 * alone; batched ones between a network's transforms. Of both, gemm_tiles.hpp takes its ranges first: plain batches of 256 to 768-byte rows from one or two such tiles
	 * per unit on, products with bias from 1 to 1.75. What its limits in bytes leave has many tiles and goes on to the streaming kernel; the limits here
	 * are for the rest: alpha or activations that have no fixed epilogue, columns that are no multiple of 16 bytes, few columns. Streaming kernel / this one, and the
	 * number of tiles:
	 *   128-byte rows  single 4: 14400 x 256 (900) 7.2 / 6.8, 20000 x 256 (1252) 7.5 / 7.9; batched 3: 15x15 1280 rows x 36 (720)
	 *                  17.9 / 17.8, 1536 (864) 19.1 / 19.7; by rows as long as that order is for (with transforms of the same order: 1024 rows of
	 *                  64 channels 15.2 / 11.9, 2048 21.1 / 15.1, 4096 25.7 / 22.5)
	 *   256-byte rows  single 4: 1024 to 1280 tiles 0.84 of the streaming kernel's time, 1280 to 1536 level; batched 3: 15x15 512 rows x 36
	 *                  (576) 17.3 / 16.5, 640 (720) 18.1 / 18.5, 896 (1008) 20.2 / 21.8, 19x19 625 (720) 22.7 / 22.2, 875 24.5 / 25.8
	 *   512-byte rows  single 5.75: 5400 x 1024 (1360) 12.7 / 11.6, 23104 x 256 with residual (1444) 17.6 / 16.0, without 13.2 / 13.9,
	 *                  24000 x 256 (1500) 13.3 / 14.3; where the streaming kernel's 128 columns are not all used, 8: 57600 x 100 (1800)
	 *                  18.7 / 16.5; batched 7: 15x15 640 rows x 36 (1440) 27.0 / 26.6, 768 (1728) 28.0 / 29.7, 896 (2016) 28.7 / 30.9,
	 *                  19x19 625 (1440) 31.2 / 29.5, 750 (1728) 32.9 / 31.0, 875 (2016) 34.2 / 34.2
	 *   768-byte rows  3: 15x15 192 rows x 36 (648) 24.0 / 21.9, 256 (864) 24.3 / 24.8; single products cross at 768 to 1024
	 *   384-byte rows  whatever gemm_tiles.hpp has left: the streaming kernel does not take them, and the tile engine, for whose pipeline 3 pieces of K are
	 *                  short, is behind or level throughout (1280 rows x 36 39.4 / 28.9; alone 32768 x 36 391 / 352, single products of
	 *                  2000 to 92000 tiles 0.55 to 0.95 of its time, below 2000 level)
	 */
	inline bool gemm_direct_applies(const StreamGemmArgs &g)
	{
		const long long tiles = static_cast<long long>(ceil_div(g.M, 64)) * ceil_div(g.N, 64) * g.batch, units = device_compute_units();
		const bool batched = g.batch > 1;
		if (g.a_row_bytes > 0xffffffffULL)
			return false;
		switch (g.k_bytes)
		{
			case 128:
				return tiles <= (batched ? 3 : 4) * units || products_meet_in_l2(g, sizeof(half_t));
			case 256:
				return tiles <= (batched ? 3 : 4) * units;
			case 384:
				return tiles <= 0xffffffffLL / 512; /* threads that a launch can have */
			case 512:
				return 4 * tiles <= (batched ? 28 : (g.N % 128 == 0) ? 23 : 32) * units;
			case 768:
				return tiles <= 3 * units;
			default:
				return false;
		}
	}
	template<int KB, typename Epilogue>
	inline void launch_gemm_direct_kb(hipStream_t stream, const StreamGemmArgs &g, const Epilogue &epilogue)
	{
		/*
		 * 64 x 64 tiles once they fill every compute unit twice, at one tile each the smaller shape is level or faster (256 rows x 36 of 128
		 * channels, 288 tiles: 4.5 against 4.8 us). 512-byte rows, of whose tiles two are resident: from 1.5 on (192 rows x 36 with the
		 * transform, 432 tiles: 17.9 against 16.8 us); 768-byte rows, of which one is, not earlier (96 x 36, 432 tiles: 6.6 against 7.5 us). By rows the
		 * loads are short and the smaller shape stays ahead to twice as many (128-byte rows, 960 rows x 36, 540 tiles, with the transform: 12.6
		 * against 12.4 us, 1408 14.2 / 13.9, 1616 14.9 / 14.9, 3072 19.1 / 19.6).
		 */
		const long long tiles = static_cast<long long>(ceil_div(g.M, 64)) * ceil_div(g.N, 64) * g.batch;
		if (2 * tiles >= (products_meet_in_l2(g, sizeof(half_t)) ? 8LL : KB == 512 ? 3LL : 4LL) * device_compute_units())
			launch_gemm_direct_as<KB, 1, 2, 4, 2>(stream, g, epilogue);
		else
			launch_gemm_direct_as<KB, 1, 1, 2, 2>(stream, g, epilogue);
	}
	template<typename Epilogue>
	inline void launch_gemm_direct(hipStream_t stream, const StreamGemmArgs &g, const Epilogue &epilogue)
	{
		switch (g.k_bytes)
		{
			case 128:
				launch_gemm_direct_kb<128>(stream, g, epilogue);
				break;
			case 256:
				launch_gemm_direct_kb<256>(stream, g, epilogue);
				break;
			case 384:
				launch_gemm_direct_kb<384>(stream, g, epilogue);
				break;
			case 512:
				launch_gemm_direct_kb<512>(stream, g, epilogue);
				break;
			case 768:
				launch_gemm_direct_kb<768>(stream, g, epilogue);
				break;
			default:
				fail_logic("HIP backend: direct GEMM: unsupported K row length");
		}
	}
} /* namespace mlhip */

#endif /* MINML_AMD_GEMM_DIRECT_HPP_ */
