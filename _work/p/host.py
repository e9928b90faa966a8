import sys, torch, time, cProfile, pstats
sys.path.insert(0,'.')
from perf import cases
c=[c for c in cases.listed() if c['name']==sys.argv[1]][0]
s=cases.prepare(c,1)
for _ in range(10): cases.run(s)
torch.cuda.synchronize()
n=200
t=time.perf_counter()
for _ in range(n): cases.run(s)
th=time.perf_counter()-t
torch.cuda.synchronize()
tt=time.perf_counter()-t
print('host us/pass',th/n*1e6,'total',tt/n*1e6)
# host alone: sync each
h=0
for _ in range(50):
    torch.cuda.synchronize(); t=time.perf_counter(); cases.run(s); h+=time.perf_counter()-t
print('host only after sync',h/50*1e6)
p=cProfile.Profile(); p.enable()
for _ in range(100): cases.run(s)
p.disable(); torch.cuda.synchronize()
pstats.Stats(p).sort_stats('tottime').print_stats(28)
